"""The tile GEMM where each k is looked up (K modes without a common base per K-tile): K in short slices, the
large tiles with their K offsets in the LDS padding, and short K on both sides of the tile shapes' lines.

Against numpy in 64 bits; sums of at most 2000 products, the tolerances of the tile kernels' other tests.
"""
import numpy as np
import pytest

import muscle
from tests.gpu_util import TOL, dev_tensor, host, randn, rel_err

pytestmark = pytest.mark.gpu

TYPES = [(np.complex128, np.complex128), (np.float64, np.float64), (np.complex64, np.complex64),
         (np.float32, np.float32), (np.float64, np.complex128), (np.complex64, np.float32)]


def _check(ta, tb, m, n, ext, a_labels, b_labels):
    """A (i and the K modes k, l) times B (the K modes and j), stored in the orders given."""
    rng = np.random.default_rng(m + n)
    size = dict(k=ext[0], l=ext[1], i=m, j=n)
    A, B = (randn(rng, [size[x] for x in lab], t) for lab, t in ((a_labels, ta), (b_labels, tb)))
    c = muscle.binary_einsum(dev_tensor(A, list(a_labels)), dev_tensor(B, list(b_labels)), out=["i", "j"])
    assert muscle.last_info()["kernel"] == 1
    got = host(c)
    wide = np.complex128 if np.iscomplexobj(got) else np.float64
    am = np.transpose(A, [a_labels.index(x) for x in "ikl"]).reshape(m, -1).astype(wide)
    bm = np.transpose(B, [b_labels.index(x) for x in "klj"]).reshape(-1, n).astype(wide)
    assert rel_err(got, am @ bm) <= TOL[got.dtype.type]


@pytest.mark.parametrize("ta, tb", TYPES, ids=lambda t: t.__name__)
@pytest.mark.parametrize("a_labels, b_labels", [("kil", "ljk"), ("ikl", "kjl")])
@pytest.mark.parametrize("m, n, ext", [
    (512, 500, (6, 85)),  # K = 510 in slices of 48, the last of 30
    (300, 400, (6, 42)),  # fewer than 256 tiles and slices
    (40, 4100, (6, 85)),  # a side below 64
    (250, 260, (3, 643)),  # K = 1929 in long slices
], ids=str)
def test_slices(m, n, ext, a_labels, b_labels, ta, tb):
    _check(ta, tb, m, n, ext, a_labels, b_labels)


@pytest.mark.parametrize("ta, tb", TYPES, ids=lambda t: t.__name__)
@pytest.mark.parametrize("a_labels, b_labels", [("kil", "ljk"), ("ikl", "kjl")])
@pytest.mark.parametrize("m, n, ext", [
    (1610, 1700, (6, 15)),  # 702 tiles, several K-tiles and a tail
    (1980, 2040, (6, 11)),  # 992 tiles
    (2040, 2100, (3, 13)),  # 1056 tiles
], ids=str)
def test_whole_k(m, n, ext, a_labels, b_labels, ta, tb):
    _check(ta, tb, m, n, ext, a_labels, b_labels)


@pytest.mark.parametrize("ta, tb", TYPES, ids=lambda t: t.__name__)
@pytest.mark.parametrize("m, n, k", [(1300, 1290, 17), (1200, 1300, 32), (1500, 1710, 24), (70000, 3, 24), (9000, 40, 31)],
                         ids=str)
def test_short_k(m, n, k, ta, tb):
    _check(ta, tb, m, n, (k, 1), "ikl", "klj")
