"""Where the power-of-two kernel's 32-bit offsets end: tensors of modes of two that lie over more than 4 GiB.

Sums of four products: the tolerances of the other contraction tests (1e-12 and 2e-5) hold with room.
"""
import numpy as np
import pytest
import torch

import muscle
from muscle.batch import ContractionBatch
from tests.gpu_util import NP2TORCH, TOL, rel_err

pytestmark = pytest.mark.gpu


def _gate(T, wide, m=1 << 16):
    """A two-site gate on m x 2 x 2 elements, the new sites last; the two new sites of the output (wide = "c")
    or the gate's own modes (wide = "b") 4 and 8 GiB apart.  Returns a, b, c, c's storage and the exact result."""
    far = (1 << 32) // np.dtype(T).itemsize
    g = torch.Generator(device="cuda").manual_seed(31)

    def tensor(extents, strides):
        size = 1 + sum((e - 1) * s for e, s in zip(extents, strides))
        flat = torch.zeros(size, dtype=NP2TORCH[T], device="cuda")
        return flat, torch.as_strided(flat, extents, strides)

    _, a = tensor([m, 2, 2], [1, m, 2 * m])
    _, b = tensor([2, 2, 2, 2], [1, 2, far, 2 * far] if wide == "b" else [1, 2, 4, 8])
    flat, c = tensor([m, 2, 2], [1, far, 2 * far] if wide == "c" else [1, m, 2 * m])
    for x in (a, b):
        x.copy_(torch.randn(x.shape, dtype=x.dtype, device="cuda", generator=g))
    wide_t = np.complex128 if np.iscomplexobj(np.zeros(1, T)) else np.float64
    ref = np.matmul(a.cpu().numpy().reshape(m, 4).astype(wide_t), b.cpu().numpy().reshape(4, 4).T.astype(wide_t))
    t = lambda x, labels: muscle.Tensor(x, list(labels))  # noqa: E731
    return t(a, "mkl"), t(b, "ijkl"), t(c, "mij"), flat, ref


@pytest.mark.parametrize("batched", [False, True], ids=["plain", "batch"])
@pytest.mark.parametrize("wide", ["c", "b"])
@pytest.mark.parametrize("T", [np.complex128, np.float32])
def test_tile_over_4_gib(T, wide, batched):
    a, b, c, flat, ref = _gate(T, wide)
    if batched:
        ContractionBatch([(c, a, b)]).run()
    else:
        muscle.binary_einsum_(c, a, b)
    torch.cuda.synchronize()
    assert rel_err(c.parent().cpu().numpy().reshape(ref.shape), ref) <= TOL[T]
    # nothing else in the output's storage was written
    assert int(torch.count_nonzero(flat)) == int(np.count_nonzero(c.parent().cpu().numpy()))


@pytest.mark.parametrize("batched", [False, True], ids=["plain", "batch"])
@pytest.mark.parametrize("shape", [(1 << 16, 4), (1 << 18, 1), (1 << 10, 1 << 10)], ids=str)
@pytest.mark.parametrize("T", [np.complex128, np.float32])
def test_empty_sum(T, shape, batched):
    """Sizes that the power-of-two kernel would take, but for a contracted mode without elements: zeros,
    in every element of an output that starts as NaN."""
    m, n = shape
    t = lambda size, labels: muscle.Tensor(  # noqa: E731
        torch.full(size, float("nan"), dtype=NP2TORCH[T], device="cuda"), list(labels))
    a, b, c = t((m, 0, 2), "ikl"), t((0, 2, n), "klj"), t((m, n), "ij")
    if batched:  # beside a pair that the power-of-two kernel does take
        x = torch.ones(2, 1 << 5, dtype=NP2TORCH[T], device="cuda")
        y = torch.ones(1 << 15, 2, dtype=NP2TORCH[T], device="cuda")
        z = t((1 << 15, 1 << 5), "ji")
        ContractionBatch([(c, a, b), (z, muscle.Tensor(x, list("ki")), muscle.Tensor(y, list("jk")))]).run()
    else:
        muscle.binary_einsum_(c, a, b)
    torch.cuda.synchronize()
    assert torch.equal(c.parent(), torch.zeros_like(c.parent()))
    if batched:
        assert torch.equal(z.parent(), torch.full_like(z.parent(), 2))
