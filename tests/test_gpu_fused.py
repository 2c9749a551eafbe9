"""MB-pol's one-launch evaluation (the default) at the edges of its blocks of 64 n-mers, against the separate
launches of the same split (the same polynomial gradients bit for bit)."""
import numpy as np
import pytest

from mbx_amd import configs, engine

pytestmark = pytest.mark.gpu

# The chain rules round differently: at most 36 terms of |k x dP/dx| < 1e3 an n-mer, four roundings each,
# 1e3 * 36 * 4 * 1.1e-16 = 1.6e-11 in one component, and some ten n-mers that come near it.
G_ABS = 1e-10


def _cluster(k, seed):
    """The k waters nearest to one of the liquid configuration's, whole molecules."""
    xyz = configs.build(configs.C1)[0].reshape(-1, 3, 3)
    o = xyz[:, 0]
    near = np.argsort(((o - o[seed]) ** 2).sum(1), kind="stable")[:k]
    return xyz[near].reshape(-1)


@pytest.mark.parametrize("box", [None, [30.0, 0, 0, 2.0, 29.0, 0, -1.0, 3.0, 31.0]], ids=["free", "triclinic"])
@pytest.mark.parametrize("waters, copies", [(3, 1), (3, 21), (3, 22), (3, 63), (3, 64), (3, 65), (12, 1), (12, 3)])
def test_block_edges(waters, copies, box):
    """copies clusters of 3 waters: 1, 63, 64, 65 trimers, 3, 63, 66, 192 dimers; 12 waters: 220 trimers of
    one first monomer after the other."""
    parts = [_cluster(waters, 3 * k) for k in range(copies)]
    if box:  # molecules of one cluster on both sides of the cell's faces
        b = np.array(box).reshape(3, 3)
        for k, p in enumerate(parts):
            w = p.reshape(-1, 3, 3)
            w -= w[0, 0] - 0.1
            w += (np.arange(waters) % 3 - 1)[:, None, None] * b[k % 3]
    out = []
    for fuse in (1, 0):
        print("fuse_chain", fuse, waters, copies, flush=True)
        e = engine.water_engine(waters * copies, box, 9.0, 6.0)
        e.set_batch(np.arange(copies + 1) * waters)
        e.set_tuning("split_3b", 4)
        e.set_tuning("fuse_chain", fuse)
        e.set_coords(np.concatenate(parts))
        e.compute()
        d, t = e.lists()
        assert len(t) == copies and len(d) == 3 * copies if waters == 3 else len(t) > 64
        out.append((e.batch_results(), e.results()))
    (ab, a), (bb, b) = out
    for k in range(2):
        np.testing.assert_allclose(ab[k], bb[k], rtol=1e-12, atol=1e-13)
    np.testing.assert_allclose(a[2], b[2], rtol=0, atol=G_ABS)
    # the virial: a sum of coordinates (up to 60 A from the origin) times such components
    np.testing.assert_allclose(ab[2], bb[2], rtol=0, atol=60 * 9 * waters * G_ABS)
    assert np.abs(a[2]).max() > 0.1
