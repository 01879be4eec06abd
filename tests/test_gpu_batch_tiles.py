"""The batched tiles' K addressing at its edges, against the oracle: K of whole and of broken K-tiles, modes
that do and do not split at one, every tile shape, whole and sliced K, a kept mode.

Sums of at most 1024 products: the tolerances of the tile kernels hold with room.
"""
import numpy as np
import pytest
import torch

import muscle
from muscle.batch import ContractionBatch
from oracle import backend_base as bb
from tests.gpu_util import NP2TORCH, TOL, dev_tensor, host, randn, rel_err

pytestmark = pytest.mark.gpu

# extents of K's modes in A's order, and B's order of them
KMODES = [((32,), (0,)), ((40,), (0,)), ((16, 3), (1, 0)), ((3, 16), (0, 1)), ((4, 2, 2, 3), (0, 1, 2, 3)),
          ((2, 8, 4), (2, 0, 1)), ((5, 8), (1, 0)), ((512,), (0,)), ((16, 33), (0, 1)), ((8, 64), (1, 0))]


SHAPES = [(70, 131), (33, 300), (300, 33), (30, 40)]  # the last one of few enough tiles to slice a long K


@pytest.mark.parametrize("T", [np.complex128, np.float64, np.complex64, np.float32])
@pytest.mark.parametrize("k_first", [True, False], ids=["kmajor", "mmajor"])
def test_k_addressing(k_first, T):
    rng = np.random.default_rng(51)
    pairs, refs, tiles = [], [], []
    for i, (ext, order) in enumerate(KMODES):
        for j, (m, n) in enumerate(SHAPES):
            ks = [f"k{x}" for x in range(len(ext))]
            se = dict(zip(ks, ext), i=m, l=n, h=2)
            ia = ks + ["i", "h"] if k_first else ["h", "i"] + ks
            ib = ["l", "h"] + [ks[x] for x in order] if k_first else [ks[x] for x in order] + ["l", "h"]
            ic = ["h", "l", "i"] if (i + j) % 2 else ["i", "l", "h"]
            A, B = randn(rng, [se[x] for x in ia], T), randn(rng, [se[x] for x in ib], T)
            C = torch.zeros([se[x] for x in reversed(ic)], dtype=NP2TORCH[T], device="cuda").permute(2, 1, 0)
            pairs.append((muscle.Tensor(C, ic), dev_tensor(A, ia), dev_tensor(B, ib)))
            wide = np.complex128 if np.iscomplexobj(A) else np.float64
            refs.append(bb.binary_einsum_general(ic, A.astype(wide), ia, B.astype(wide), ib))
            tiles.append(j % 3)
    batch = ContractionBatch(pairs, tiles=tiles)
    routes = {batch.pair_info(i)["route"] for i in range(len(pairs))}
    assert "tiles" in routes and "split_k" in routes
    batch.run()
    for (c, _, _), ref in zip(pairs, refs):
        assert rel_err(host(c), ref) <= TOL[T]
