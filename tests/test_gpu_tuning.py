"""The schedule switches (mbxg_set_tuning, mbxg_autotune): what was not timed or asked for stays as it was."""
import numpy as np
import pytest

from conftest import water_case
from mbx_amd import engine

pytestmark = pytest.mark.gpu


def _water(systems, key="h2o_256_cubic"):
    xyz, box, c2, c3, _ = water_case(systems, key)
    e = engine.water_engine(len(xyz) // 9, box, c2, c3)
    e.set_coords(xyz)
    return e


def _droplet(systems, n):
    """The n waters of the liquid nearest to its first one, in the gas phase."""
    xyz = water_case(systems, "h2o_256_cubic")[0].reshape(-1, 3, 3)
    near = np.argsort(((xyz[:, 0] - xyz[0, 0]) ** 2).sum(1), kind="stable")[:n]
    e = engine.water_engine(n, None, 9.0, 6.0)
    e.set_coords(xyz[near].reshape(-1))
    return e


def _separate_ms(e):
    """The shortest time of the stages that are launches of their own only without the one launch."""
    e.set_timing(True)
    out = []
    for _ in range(6):
        e.compute()
        t = e.timings()
        out.append(t["vars_3b"] + t["chain_3b"] + t["chain_2b"])
    e.set_timing(False)
    return min(out[1:])


def test_untimed_2b_split_stays(systems):
    """On the paired path the 2B polynomial has no time of its own: its split stays with the rule."""
    e = _water(systems)
    e.compute()
    before = e.tuning("split_2b")
    assert e.autotune(reps=1)["split_2b"] == before


@pytest.mark.parametrize("terms", [engine.TERM_2B | engine.TERM_3B, engine.TERM_3B])
def test_other_computes_keep_the_one_launch(systems, terms):
    """Tuned for energies (of few n-mers, which eight wavefronts do fastest), a compute of both orders with
    gradients still is one launch."""
    e = _droplet(systems, 40)
    e.compute()
    e.set_tuning("fuse_chain", 0)
    separate = _separate_ms(e)
    e.set_tuning("fuse_chain", 1)
    assert _separate_ms(e) < 0.5 * separate
    e.autotune(terms=terms, do_grads=False, reps=3)
    assert e.tuning("fuse_chain") == 1
    assert _separate_ms(e) < 0.5 * separate


def test_autotune_error_restores(systems):
    """A refused compute (the 1B term over a batch) leaves schedule and timing as they were."""
    xyz, box, c2, c3, _ = water_case(systems, "h2o_256_cubic")
    n = len(xyz) // 9
    e = engine.water_engine(2 * n, box, c2, c3)
    e.set_batch([0, n, 2 * n])
    e.set_coords(np.concatenate([xyz, xyz]))
    e.compute()
    keys = ("split_2b", "split_3b", "split_ch4h2o2_3b", "fuse_poly", "fuse_chain", "fuse_vars")
    before = {k: e.tuning(k) for k in keys}
    with pytest.raises(engine.MbxgError):
        e.autotune(terms=engine.TERM_1B | engine.TERM_2B | engine.TERM_3B, reps=1)
    assert {k: e.tuning(k) for k in keys} == before
    e.compute()
    with pytest.raises(engine.MbxgError):
        e.timings()


def test_back_to_the_rule(systems):
    """0 gives a split back to the rule; what tuning() returns by default can be set without a change of route."""
    e = _water(systems)
    e.compute()
    default = {k: e.tuning(k) for k in ("split_2b", "split_3b")}
    for k in default:
        e.set_tuning(k, 1)
        assert e.tuning(k) == 1
        e.set_tuning(k, 0)
        assert e.tuning(k) == default[k]
    e.set_tuning("fuse_chain", 0)
    separate = _separate_ms(e)
    e.set_tuning("fuse_chain", 1)
    e.set_tuning("split_3b", default["split_3b"])
    assert _separate_ms(e) < 0.5 * separate
    with pytest.raises(engine.MbxgError):
        e.set_tuning("split_ch4h2o2_3b", 0)


def test_autotuned_schedule_is_replayed(systems):
    """A step captured before the autotuner ran is captured again: same results as an eager compute of the
    schedule found."""
    e = _water(systems)
    e.set_graph(True)
    for _ in range(3):
        e.compute()
    e.results()
    e.autotune(reps=1)
    first = e.results()
    for _ in range(3):
        e.compute()
        again = e.results()
        assert again[:2] == first[:2]
        np.testing.assert_allclose(again[2], first[2], rtol=0, atol=1e-9)
