"""The power-of-two kernel at its edges, against the oracle: one tile to several per workgroup, every
split of the tile between the operands, one K chunk and many, and the forms it leaves to the others.

Sums of at most 128 products: the tolerances of the tile kernels (1e-12 and 2e-5) hold with room.
"""
import random

import numpy as np
import pytest
import torch

import muscle
from muscle.batch import ContractionBatch
from tests.gpu_util import NP2TORCH, TOL, rel_err

pytestmark = pytest.mark.gpu

TYPES = [np.complex128, np.float64, np.complex64, np.float32]
# log2 of M, N, K and the kept modes' extent
PLAIN = [(5, 6, 3, 0), (6, 6, 4, 0), (12, 6, 2, 0), (9, 9, 1, 0), (7, 7, 2, 4), (6, 5, 3, 2), (0, 18, 2, 0), (18, 1, 3, 0),
         (2, 18, 7, 0), (17, 3, 5, 0), (3, 14, 5, 3), (11, 12, 2, 0), (10, 8, 3, 5)]
BATCHED = [(9, 9, 1, 0), (10, 8, 2, 0), (6, 11, 3, 0), (5, 12, 4, 0), (0, 17, 2, 0), (3, 15, 5, 0), (14, 4, 7, 0),
           (4, 10, 6, 3), (7, 7, 4, 3), (11, 12, 2, 0), (6, 6, 1, 0), (12, 5, 9, 0)]


def _pair(case, T, seed, gaps=False):
    """Device operands of 2-, 4- and 8-valued modes in a random order, in storage of another random order
    (with gaps between the elements if asked), an output of the same kind and the exact result."""
    rng = random.Random(seed)
    nxt = iter(range(10000))
    ext = {}

    def modes(bits, kind):
        out = []
        while bits:
            w = min(bits, rng.choice([1, 1, 2, 3]))
            out.append(f"{kind}{next(nxt)}")
            ext[out[-1]] = 1 << w
            bits -= w
        return out

    m, n, k, h = (modes(b, c) for b, c in zip(case, "mnkh"))
    g = torch.Generator(device="cuda").manual_seed(seed)

    def tensor(labels, fill):
        inds, store = list(labels), list(labels)
        rng.shuffle(inds)
        rng.shuffle(store)
        stride, s = {}, 1
        for x in store:
            if gaps and rng.random() < 0.2:
                s *= rng.choice([2, 3])
            stride[x] = s
            s *= ext[x]
        flat = torch.zeros(s, dtype=NP2TORCH[T], device="cuda")
        if fill:
            flat = torch.randn(s, dtype=NP2TORCH[T], device="cuda", generator=g)
        return muscle.Tensor(torch.as_strided(flat, [ext[x] for x in inds], [stride[x] for x in inds]), inds)

    a, b, c = tensor(m + k + h, True), tensor(k + n + h, True), tensor(m + n + h, False)

    def matrix(t, rows, cols):
        inds = [i.tag for i in t.inds()]
        perm = [inds.index(x) for x in h + rows + cols]
        size = [int(np.prod([ext[x] for x in y])) for y in (h, rows, cols)]
        return t.parent().cpu().permute(perm).reshape(size).numpy()

    wide = np.complex128 if np.iscomplexobj(np.zeros(1, T)) else np.float64
    ref = np.matmul(matrix(a, m, k).astype(wide), matrix(b, k, n).astype(wide))
    return a, b, c, lambda: rel_err(matrix(c, m, n), ref)


@pytest.mark.parametrize("T", TYPES)
@pytest.mark.parametrize("gaps", [False, True], ids=["dense", "gaps"])
@pytest.mark.parametrize("case", PLAIN, ids=str)
def test_plain(case, gaps, T):
    a, b, c, err = _pair(case, T, sum(case) + 100, gaps)
    muscle.binary_einsum_(c, a, b)
    torch.cuda.synchronize()
    if case[3] == 0:  # kept modes may fill C's lowest bits, and leave a pair to the tile GEMM
        assert muscle.last_info()["kernel"] == 2
    assert err() <= TOL[T]


@pytest.mark.parametrize("T", TYPES)
@pytest.mark.parametrize("gaps", [False, True], ids=["dense", "gaps"])
def test_batched(gaps, T):
    """All in one launch, beside pairs that other kernels take (64 tiles of the kernel are its least)."""
    pairs = [_pair(case, T, i + 500, gaps) for i, case in enumerate(BATCHED)]
    batch = ContractionBatch([(c, a, b) for a, b, c, _ in pairs])
    for mode in ("persistent", "persistent_nograph", "persistent"):
        for p in pairs:
            p[2].parent().zero_()
        batch.run(mode)
        torch.cuda.synchronize()
        for case, p in zip(BATCHED, pairs):
            assert p[3]() <= TOL[T], case
    for i, case in enumerate(BATCHED):
        k, side = 1 << case[2], 1 << min(case[:2])
        if k <= 16 and side > 16:
            assert batch.pair_info(i)["route"] == "shallow"


@pytest.mark.parametrize("shape", [(3 << 9, 1 << 9, 2), (1 << 10, 1 << 9, 3), (1 << 10, 130, 4)], ids=str)
def test_other_extents(shape):
    """An extent that is no power of two leaves the contraction to the other kernels."""
    m, n, k = shape
    g = torch.Generator(device="cuda").manual_seed(7)
    a = torch.randn(m, k, dtype=torch.complex128, device="cuda", generator=g)
    b = torch.randn(k, n, dtype=torch.complex128, device="cuda", generator=g)
    c = muscle.binary_einsum(muscle.Tensor(a, ["i", "k"]), muscle.Tensor(b, ["k", "l"]))
    batch_out = muscle.Tensor(torch.zeros(m, n, dtype=torch.complex128, device="cuda"), ["i", "l"])
    ContractionBatch([(batch_out, muscle.Tensor(a, ["i", "k"]), muscle.Tensor(b, ["k", "l"]))]).run()
    torch.cuda.synchronize()
    ref = a.cpu().numpy() @ b.cpu().numpy()
    assert rel_err(c.parent().cpu().numpy(), ref) <= TOL[np.complex128]
    assert rel_err(batch_out.parent().cpu().numpy(), ref) <= TOL[np.complex128]
