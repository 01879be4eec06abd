"""The tile GEMM's shapes and K addressing at their edges, against the oracle.

Every element type runs the large tiles (1024 and more 64 x 64 tiles; 2048 for
complex FP64) and the small ones, with M and N off the tile edges, K below, at
and past a K-tile, and K made of several modes whose offsets do and do not
split at the K-tile (one base per tile, or a lookup per k).
"""
import numpy as np
import pytest

import muscle
from oracle import backend_base as bb
from tests.gpu_util import TOL, dev_tensor, host, randn, rel_err

pytestmark = pytest.mark.gpu

# K modes (extents, in A's order) and B's order of them
KMODES = [((8,), (0,)), ((9,), (0,)), ((16,), (0,)), ((47,), (0,)), ((16, 3), (1, 0)), ((8, 5), (0, 1)), ((3, 13), (1, 0)),
          ((2, 3, 2, 7), (3, 1, 0, 2)), ((4, 2, 2, 5), (2, 0, 3, 1))]


def _check(T, ia, sa, ib, sb, ic, kernel=1):
    rng = np.random.default_rng(41)
    A, B = randn(rng, sa, T), randn(rng, sb, T)
    c = muscle.binary_einsum(dev_tensor(A, ia), dev_tensor(B, ib), out=ic)
    assert muscle.last_info()["kernel"] == kernel
    got = host(c)
    wide = np.complex128 if np.iscomplexobj(A) else np.float64
    ref = bb.binary_einsum_general(ic, A.astype(wide), ia, B.astype(wide), ib)
    assert rel_err(got, ref) <= TOL[T], rel_err(got, ref)


@pytest.mark.parametrize("T", [np.complex128, np.float64, np.complex64, np.float32])
@pytest.mark.parametrize("k_first", [True, False], ids=["kmajor", "mmajor"])
@pytest.mark.parametrize("kmodes", KMODES, ids=lambda k: "x".join(map(str, k[0])))
def test_small_tiles(kmodes, k_first, T):
    ext, order = kmodes
    ks = [f"k{i}" for i in range(len(ext))]
    kb = [ks[i] for i in order]
    se = dict(zip(ks, ext), i=70, l=131)
    ia = ks + ["i"] if k_first else ["i"] + ks
    ib = kb + ["l"] if not k_first else ["l"] + kb
    _check(T, ia, [se[x] for x in ia], ib, [se[x] for x in ib], ["i", "l"])


@pytest.mark.parametrize("T, m, n", [(np.complex128, 2890, 2951), (np.float64, 2050, 2111), (np.complex64, 2050, 2111),
                                     (np.float32, 2050, 2111)])
@pytest.mark.parametrize("ext, order", [((40,), (0,)), ((37,), (0,)), ((3, 13), (1, 0)), ((16, 3), (1, 0))],
                         ids=lambda e: "x".join(map(str, e)))
def test_large_tiles(ext, order, T, m, n):
    ks = [f"k{i}" for i in range(len(ext))]
    se = dict(zip(ks, ext), i=m, l=n)
    ia, ib = ["i"] + ks, [ks[i] for i in order] + ["l"]
    _check(T, ia, [se[x] for x in ia], ib, [se[x] for x in ib], ["l", "i"])


@pytest.mark.parametrize("k", [1024, 1031])
@pytest.mark.parametrize("mult", [3, 4])
def test_long_k_complex_fp64(k, mult):
    with muscle.with_backend(muscle.BackendHIP(complex_mult=mult)):
        _check(np.complex128, ["k", "i"], (k, 2890), ["l", "k"], (2951, k), ["i", "l"])


@pytest.mark.parametrize("ta, tb", [(np.float64, np.complex128), (np.complex64, np.float32)])
@pytest.mark.parametrize("m, n, k", [(70, 131, 45), (2050, 2111, 45)])
def test_real_by_complex(ta, tb, m, n, k):
    rng = np.random.default_rng(42)
    A, B = randn(rng, (m, k), ta), randn(rng, (k, n), tb)
    c = muscle.binary_einsum(dev_tensor(A, ["i", "k"]), dev_tensor(B, ["k", "l"]))
    ref = A.astype(np.complex128) @ B.astype(np.complex128)
    assert rel_err(host(c), ref) <= TOL[np.dtype(host(c).dtype).type]


def test_batched_tiles_and_negative_span():
    """A kept mode beside ragged tiles, and operands that are reversed views (their lowest offset is
    not the first element's)."""
    import ctypes

    import torch

    from muscle import _lib
    from muscle.ops import _handle_for
    rng = np.random.default_rng(43)
    A, B = randn(rng, (70, 40, 3), np.complex128), randn(rng, (40, 99, 3), np.complex128)
    c = muscle.binary_einsum(dev_tensor(A, ["i", "k", "h"]), dev_tensor(B, ["k", "l", "h"]), out=["i", "l", "h"])
    ref = np.einsum("ikh,klh->ilh", A, B)
    assert rel_err(host(c), ref) <= TOL[np.complex128]

    a, b = dev_tensor(A[:, :, 0], ["i", "k"]), dev_tensor(B[:, :, 0], ["k", "l"])
    out = torch.zeros(99, 70, dtype=torch.complex128, device="cuda")  # column-major (70, 99)
    # A with both modes reversed, B with k reversed: the same products over k
    da = _lib.Desc(_lib.C64, a.parent().data_ptr() + 16 * (70 * 40 - 1), [1, 2], [70, 40], [-1, -70])
    db = _lib.Desc(_lib.C64, b.parent().data_ptr() + 16 * 39, [2, 3], [40, 99], [-1, 40])
    dc = _lib.Desc(_lib.C64, out.data_ptr(), [1, 3], [70, 99], [1, 70])
    h = _handle_for(0)
    info = _lib.Info()
    _lib.check(_lib.lib.muscle_hip_binary_einsum(h, dc.ref, da.ref, db.ref, 0, 1e-12, ctypes.byref(info)))
    torch.cuda.synchronize()
    assert info.kernel == 1
    assert rel_err(out.cpu().numpy().T, A[::-1, :, 0] @ B[:, :, 0]) <= TOL[np.complex128]
