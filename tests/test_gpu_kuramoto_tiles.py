"""The Kuramoto kernel's tiles (nemosim_amd/plugins/Kuramoto.hip) at their
edges, bit for bit against the oracle: workgroups of 768, 2304 and 4608
couplings, up to 16 oscillators of a workgroup and more, rows that end on them and one past them (read in pieces), several
tiles in one workgroup where rows are uneven, rows around the sums' steps of
32 and 64 terms, and empty rows."""
import numpy as np
import pytest

from test_gpu_kuramoto import Pair

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129]


def uneven(n, seed):
    """about 10 couplings each, the steps' edges, and neighbours that do not
    share a tile of 768 (500 and 500; 700 and 69; 768; 769; 1537)"""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 20, n)
    deg[:len(EDGES)] = EDGES
    deg[100:110] = [500, 500, 700, 69, 768, 0, 769, 3, 1537, 1]
    return deg


@pytest.mark.parametrize("deg", [
    uneven(1024, 1),                                 # one oscillator per workgroup
    uneven(1025, 2),                                 # two
    uneven(5000, 3),                                 # five
    uneven(16384, 4),                                # 16, a row of lanes each
    uneven(16385, 5),                                # 17, a lane each
    np.array([2000, 2100, 1900, 2303, 2304, 2305, 2000]),    # tiles of 2304, one row past
    np.array([2400, 4608, 2304, 2305, 4609, 2200]),  # tiles of 4608, one row past
    np.array([4608, 9217, 4600]),                    # every row in pieces or a whole tile
], ids=["1024", "1025", "5000", "16384", "16385", "2304", "4608", "pieces"])
def test_tiles(nemo_mod, oracle_mod, deg):
    n = len(deg)
    rng = np.random.default_rng(n)
    nsyn = int(deg.sum())
    tgt = np.repeat(np.arange(n), deg)
    src = rng.integers(0, n, nsyn)
    order = np.argsort(src, kind="stable")
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint64)
    dly = rng.integers(1, 32, nsyn).astype(np.uint8)
    w = rng.normal(0.0, 0.05, nsyn).astype(np.float32)
    p = Pair(nemo_mod, oracle_mod, rng.uniform(0.0, 0.2, n), rng.uniform(0.0, 2 * np.pi, n),
             csr=(rowptr, tgt[order].astype(np.uint32), dly, w))
    for t in range(3):
        p.step()
    p.check(3)
