"""Performance cases of the contraction library: what its users call, over the sizes they call it with.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs (and the batch or server a program keeps) on the GPU
    run(state)          one pass through the public entry points; returns its outputs
    work(case)          bytes and flops of one pass: every input read once, every output written once
    exact(case, seed)   the outputs in 64 bits from plain torch, or None

A case is a dict of plain values.  Index labels are single letters; "spec" is an
einsum-like text ("ijk,klj->il") and "ext" gives extents ("i64 j32"; a label
that it leaves out has dimension 2).  Tensors are column-major, as the library
allocates them.  Element types: f32, f64, c32 (ComplexF32), c64 (ComplexF64).
"""
import os
import random
import string
import sys

import numpy as np
import torch

# the package of the tree this file is run in (the working folder)
sys.path.insert(0, os.path.abspath("muscle.jl_amd"))

import muscle  # noqa: E402
from muscle.batch import ContractionBatch  # noqa: E402
from muscle.serve import LeafBank, Server, tree_nodes  # noqa: E402
from muscle.workloads import circuit_pairs, contraction_tree  # noqa: E402

DTYPES = {"f32": torch.float32, "f64": torch.float64, "c32": torch.complex64, "c64": torch.complex128}
SIZES = {"f32": 4, "f64": 8, "c32": 8, "c64": 16}
LETTERS = string.ascii_letters


# ---------------------------------------------------------------- the cases
def _interleaved(d):
    """Rank-6 pair with every extent d whose contracted modes sit at positions (2, 4, 6) of A
    and (1, 3, 5) of B, output order interleaved: M = N = K = d^3, every operand permuted."""
    return "aubvcw,udvewf->adbecf", " ".join(f"{x}{d}" for x in "abcdefuvw")


def _hyper(a, c, h, b):
    """Pair with a kept (batch) index h: M = a * 2a, K = c * 2c, N = b * 2b per batch entry."""
    return "auhbv,uchvd->achbd", f"a{a} b{2 * a} u{c} v{2 * c} c{b} d{2 * b} h{h}"


def _gate(rank, qubits, at):
    """A gate on `qubits` of the `rank` two-level sites of a state vector: the contracted sites sit
    at the positions that `at` seeds; the output keeps the default order (state's sites, then the
    gate's new ones)."""
    r = random.Random(at)
    state = list(LETTERS[:rank])
    hit = r.sample(state, qubits)
    new = list(LETTERS[rank:rank + qubits])
    out = [x for x in state if x not in hit] + new
    return f"{''.join(state)},{''.join(new + hit)}->{''.join(out)}"


def _dims2(m, n, k, h, order):
    """A pair of a circuit-like network: every index of dimension 2, m / n open indices left and
    right, k contracted and h kept ones, all orders random (seeded by `order`)."""
    r = random.Random(order)
    lab = list(LETTERS[:m + n + k + h])
    left, right, con, hyp = lab[:m], lab[m:m + n], lab[m + n:m + n + k], lab[m + n + k:]
    shuf = [left + con + hyp, con + hyp + right, left + right + hyp]
    for s in shuf:
        r.shuffle(s)
    return "{},{}->{}".format(*("".join(s) for s in shuf))


def listed():
    cube, cube_ext = _interleaved(16)
    hyp, hyp_ext = _hyper(16, 16, 64, 16)
    perm = list(LETTERS[:24])
    random.Random(24).shuffle(perm)
    return [
        # the smallest calls: one small plain contraction, where launches and the host path count
        dict(name="plain_c64_64x96x1536", kind="binary", dtype="c64", spec="ijk,klj->il", ext="i64 j32 k48 l96"),
        # a two-site gate on a state vector of 22 two-level sites: a stream over the state
        dict(name="gate_c64_rank22", kind="binary", dtype="c64", spec=_gate(22, 2, 5), inplace=True),
        # two site tensors of a matrix product state joined over their bond; odd extents, real FP64
        dict(name="bond_f64_1497x1509x501", kind="binary", dtype="f64", spec="lpr,rqs->lpqs",
             ext="l499 p3 r501 q3 s503"),
        # the large GEMM-shaped contraction on permuted layouts, M = N = K = 4096
        dict(name="cube_c64_4096", kind="binary", dtype="c64", spec=cube, ext=cube_ext),
        # the same product at a stated error on the low-precision units
        dict(name="cube_c64_4096_ozaki_1e-10", kind="binary", dtype="c64", spec=cube, ext=cube_ext,
             precision="ozaki_int8", target=1e-10),
        # a kept index: 64 products of 512^3 in ComplexF32
        dict(name="hyper_c32_64x512", kind="binary", dtype="c32", spec=hyp, ext=hyp_ext),
        # one large step of a circuit network's contraction: short sum, 2^24 outputs, random mode orders
        dict(name="dims2_c64_m12_n12_k5", kind="binary", dtype="c64", spec=_dims2(12, 12, 5, 0, 7), inplace=True),
        # many uneven pairs of such networks in one launch
        dict(name="batch_c64_256", kind="batch", dtype="c64", pairs=256, rank_max=22, structure=0),
        # elementwise product with a permuted operand
        dict(name="hadamard_c64_permuted", kind="hadamard", dtype="c64", spec="ijk,kij->ijk", ext="i250 j333 k301"),
        # permutation of a rank-24 circuit tensor
        dict(name="permute_c64_rank24", kind="unary", dtype="c64", spec=f"{LETTERS[:24]}->{''.join(perm)}"),
        # the factorization behind a two-site update: theta (chi, d, d, chi) split in the middle
        dict(name="svd_c64_128", kind="svd", dtype="c64", chi=64, d=2),
        # contraction-tree jobs through the server: small trees, latency and scheduling
        dict(name="served_24_jobs", kind="served", jobs=24, size_lo=4, size_hi=16, structure=0),
    ]


def draw(rng):
    dt = rng.choice(["c64", "c64", "c32"])
    any_dt = rng.choice(["c64", "c32", "f64", "f32"])

    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["plain", "plain", "gate", "gate", "cube", "ozaki", "hyper", "dims2", "dims2", "dims2", "batch",
                       "hadamard", "unary", "sum", "svd", "served"])
    if kind == "plain":
        spec = rng.choice(["ijk,klj->il", "lpr,rqs->lpqs", "lpr,rqs->plsq", "xjk,jyk->yx"])
        joined = spec.startswith("lpr")  # two site tensors: wide bonds, narrow sites
        lim = {x: (8, 500) if joined else (8, 1500) for x in spec if x.isalpha()}
        for x in "pqjk":
            lim[x] = (2, 4) if joined else (2, 48)
        return dict(kind="binary", dtype=any_dt, spec=spec,
                    ext=" ".join(f"{x}{log_int(*lim[x])}" for x in sorted({y for y in spec if y.isalpha()})))
    if kind == "gate":
        return dict(kind="binary", dtype=dt, spec=_gate(rng.randint(8, 24), rng.randint(1, 3), rng.randint(0, 9999)),
                    inplace=True)
    if kind in ("cube", "ozaki"):
        spec, ext = _interleaved(rng.randint(6, 16))
        case = dict(kind="binary", dtype=any_dt if kind == "cube" else rng.choice(["c64", "f64"]), spec=spec, ext=ext)
        if kind == "ozaki":
            case.update(precision="ozaki_int8", target=rng.choice([1e-10, 1e-12]))
        return case
    if kind == "hyper":
        spec, ext = _hyper(rng.randint(4, 16), rng.randint(4, 16), log_int(2, 64), rng.randint(4, 16))
        return dict(kind="binary", dtype=any_dt, spec=spec, ext=ext)
    if kind == "dims2":
        m, n, k, h = rng.randint(2, 12), rng.randint(2, 12), rng.randint(1, 10), rng.randint(0, 2)
        h = min(h, 24 - m - n)
        return dict(kind="binary", dtype=dt, spec=_dims2(m, n, k, h, rng.randint(0, 9999)), inplace=True)
    if kind == "batch":
        return dict(kind="batch", dtype=dt, pairs=log_int(24, 256), rank_max=rng.randint(10, 22),
                    structure=rng.randint(1, 9999))
    if kind == "hadamard":
        spec = rng.choice(["ijk,kij->ijk", "ijk,j->ijk", "ijk,ki->ijk", "ijk,ijk->ijk"])
        return dict(kind="hadamard", dtype=any_dt, spec=spec, ext=" ".join(f"{x}{log_int(10, 330)}" for x in "ijk"))
    if kind == "unary":
        rank = rng.randint(10, 24)
        perm = list(LETTERS[:rank])
        rng.shuffle(perm)
        return dict(kind="unary", dtype=any_dt, spec=f"{LETTERS[:rank]}->{''.join(perm)}")
    if kind == "sum":
        spec = rng.choice(["ijk->k", "ijk->i", "ijk->ik", "ijk->ij", "iji->j", "iijk->jk"])
        hi = 400 if len(spec.split("->")[0]) == 3 else 90
        return dict(kind="unary", dtype=any_dt, spec=spec,
                    ext=" ".join(f"{x}{log_int(10, hi)}" for x in sorted({y for y in spec if y.isalpha()})))
    if kind == "svd":
        return dict(kind="svd", dtype=rng.choice(["c64", "f64"]), chi=log_int(8, 64), d=2)
    return dict(kind="served", jobs=log_int(2, 24), size_lo=4, size_hi=rng.randint(8, 16), structure=rng.randint(1, 9999))


# ---------------------------------------------------------------- inputs
def _parse(case):
    left, out = case["spec"].split("->")
    ext = {x: 2 for x in left if x != ","}
    for w in case.get("ext", "").split():
        ext[w[0]] = int(w[1:])
    return left.split(","), out, ext


def _count(labels, ext):
    n = 1
    for x in labels:
        n *= ext[x]
    return n


def _strides(labels, ext):
    s, out = 1, []
    for x in labels:
        out.append(s)
        s *= ext[x]
    return out


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _col_major(flat, labels, ext):
    """A tensor over `flat` (its first elements), column-major."""
    return muscle.Tensor(flat.as_strided([ext[x] for x in labels], _strides(labels, ext)), list(labels))


def _operands(case, seed):
    """Flat buffers of the inputs: iid normal, scaled so that a contraction's outputs are of unit size."""
    ins, out, ext = _parse(case)
    summed = _count({x for i in ins for x in i} - set(out), ext)
    g = _generator(seed)
    scale = summed ** (-0.25) if case["kind"] == "binary" else 1.0
    flats = []
    for i in ins:
        x = torch.randn(_count(i, ext), dtype=DTYPES[case["dtype"]], device="cuda", generator=g)
        flats.append(x.mul_(scale) if scale != 1.0 else x)
    return ins, out, ext, flats


_POOL = 1 << 23  # elements of the pool a batch's operands are views of


def _batch_structure(case):
    pairs = circuit_pairs(case["pairs"], case["structure"], ranks=(4, case["rank_max"]),
                          out_ranks=(4, min(24, case["rank_max"] + 2)))
    rng = np.random.default_rng(case["structure"] + 1)
    offs = [tuple(int(rng.integers(0, _POOL - (1 << len(x)) + 1)) for x in p[:2]) for p in pairs]
    return pairs, offs


def _batch_pool(case, seed):
    return torch.randn(_POOL, dtype=DTYPES[case["dtype"]], device="cuda", generator=_generator(seed))


def _jobs(case, seed):
    """The trees of the case's jobs, ComplexF64 and ComplexF32 in turn, and their leaves."""
    specs = [contraction_tree(case["structure"] + i, size_log2=(case["size_lo"], case["size_hi"]),
                              dtype="c64" if i % 2 == 0 else "c32") for i in range(case["jobs"])]
    bank = LeafBank(seed=seed)
    bank.reserve(specs)
    rng = np.random.default_rng(seed)
    return specs, bank, [bank.leaves(s, rng) for s in specs]


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("binary", "hadamard", "unary"):
        ins, out, ext, flats = _operands(case, seed)
        state["in"] = [_col_major(f, i, ext) for f, i in zip(flats, ins)]
        state["out"] = [muscle.Index(x) for x in out]
        if kind == "binary":
            state["backend"] = None
            if case.get("precision"):
                state["backend"] = muscle.BackendHIP(precision=case["precision"], target_rel_error=case["target"])
        if kind != "binary" or case.get("inplace"):
            state["flat"] = torch.empty(_count(out, ext), dtype=DTYPES[case["dtype"]], device="cuda")
            state["c"] = _col_major(state["flat"], out, ext)
    elif kind == "batch":
        pairs, offs = _batch_structure(case)
        pool = _batch_pool(case, seed)
        arena = torch.empty(sum(1 << len(p[2]) for p in pairs), dtype=DTYPES[case["dtype"]], device="cuda")
        ext = dict.fromkeys({x for p in pairs for t in p for x in t}, 2)
        ts, at = [], 0
        for (ia, ib, ic), (oa, ob) in zip(pairs, offs):
            ts.append((_col_major(arena[at:], ic, ext), _col_major(pool[oa:], ia, ext), _col_major(pool[ob:], ib, ext)))
            at += 1 << len(ic)
        state.update(batch=ContractionBatch(ts), pool=pool, arena=arena)
    elif kind == "svd":
        chi, d = case["chi"], case["d"]
        x = torch.randn(chi * d * d * chi, dtype=DTYPES[case["dtype"]], device="cuda", generator=_generator(seed))
        state["theta"] = _col_major(x, "lpqr", {"l": chi, "p": d, "q": d, "r": chi})
    else:
        specs, bank, leaves = _jobs(case, seed)
        server = Server(pool_gib=1.0)
        state.update(server=server, bank=bank,
                     prepared=[server.prepare(lv, tree_nodes(s)) for lv, s in zip(leaves, specs)])
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "binary":
        a, b = state["in"]
        if "c" in state:  # into the caller's tensor
            muscle.binary_einsum_(state["c"], a, b)
            return state["flat"]
        if state["backend"] is None:
            return muscle.binary_einsum(a, b, out=state["out"]).parent()
        with muscle.with_backend(state["backend"]):
            return muscle.binary_einsum(a, b, out=state["out"]).parent()
    if kind == "hadamard":
        muscle.hadamard_(state["c"], *state["in"])
        return state["flat"]
    if kind == "unary":
        muscle.unary_einsum_(state["c"], state["in"][0])
        return state["flat"]
    if kind == "batch":
        state["batch"].run()
        return state["arena"]
    if kind == "svd":
        u, s, v = muscle.tensor_svd_thin(state["theta"], inds_u=["l", "p"], inds_v=["q", "r"], ind_s="s")
        return [u.parent(), s.parent(), v.parent()]
    server = state["server"]
    ids = [server.submit_prepared(p) for p in state["prepared"]]
    roots = []
    for i in ids:
        server.wait(i)
        x = server.result(i).parent()
        roots.append(x.permute(*reversed(range(x.dim()))).reshape(-1) if x.dim() else x)  # its memory order
        server.release(i)
    return roots


# ---------------------------------------------------------------- what a pass cannot do without
def _pair_flops(dtype, points):
    return (8.0 if dtype[0] == "c" else 2.0) * points


def work(case):
    kind = case["kind"]
    if kind in ("binary", "hadamard", "unary"):
        ins, out, ext = _parse(case)
        es = SIZES[case["dtype"]]
        # a repeated label inside one operand reads its diagonal only
        elems = sum(_count(set(i), ext) for i in ins) + _count(out, ext)
        if kind == "binary":
            flops = _pair_flops(case["dtype"], _count({x for i in ins for x in i}, ext))
        elif kind == "hadamard":
            flops = (6.0 if case["dtype"][0] == "c" else 1.0) * _count(out, ext)
        else:
            flops = (2.0 if case["dtype"][0] == "c" else 1.0) * _count(set(ins[0]), ext)
            flops = flops if _count(out, ext) < _count(set(ins[0]), ext) else 0.0
        return {"bytes": float(elems * es), "flops": flops}
    if kind == "batch":
        pairs, _ = _batch_structure(case)
        es = SIZES[case["dtype"]]
        return {"bytes": float(sum(sum(1 << len(t) for t in p) for p in pairs) * es),
                "flops": sum(_pair_flops(case["dtype"], 2.0 ** len(set(p[0]) | set(p[1]))) for p in pairs)}
    if kind == "svd":
        # a thin SVD of an n x n matrix: about 20 n^3 multiply-add pairs' flops (bidiagonalisation,
        # iteration and both sets of vectors), four times that in complex arithmetic
        n = case["chi"] * case["d"]
        cplx = case["dtype"][0] == "c"
        return {"bytes": float((3 * n * n) * SIZES[case["dtype"]] + 8 * n), "flops": (4.0 if cplx else 1.0) * 20.0 * n ** 3}
    by = fl = 0.0
    for i in range(case["jobs"]):
        dtype = "c64" if i % 2 == 0 else "c32"
        spec = contraction_tree(case["structure"] + i, size_log2=(case["size_lo"], case["size_hi"]), dtype=dtype)
        labels = [set(x) for x in spec.leaves] + [set(x[2]) for x in spec.nodes]
        by += SIZES[dtype] * (sum(2.0 ** len(x) for x in spec.leaves) + 2.0 ** len(labels[-1]))
        fl += sum(_pair_flops(dtype, 2.0 ** len(labels[a] | labels[b])) for a, b, _ in spec.nodes)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------- the same in 64 bits
def _wide(x):
    return x.to(torch.complex128 if x.is_complex() else torch.float64)


def _offsets(order, labels, ext):
    """Element offsets of a column-major tensor with `labels`, over the points of `order`
    (a list of labels, the first fastest); a label repeated in `labels` adds its strides up."""
    st = {}
    for x, s in zip(labels, _strides(labels, ext)):
        st[x] = st.get(x, 0) + s
    off = torch.zeros(1, dtype=torch.int64, device="cuda")
    for x in order:
        off = (torch.arange(ext[x], device="cuda", dtype=torch.int64)[:, None] * st.get(x, 0) + off[None, :]).reshape(-1)
    return off


def _contract(a, ia, b, ib, ic, ext):
    """C (flat, column-major in ic) = sum over the labels that ic lacks, in 64 bits."""
    bat = [x for x in ic if x in ia and x in ib]
    m = [x for x in ic if x in ia and x not in ib]
    n = [x for x in ic if x in ib and x not in ia]
    k = [x for x in dict.fromkeys(ia) if x in ib and x not in ic]
    grid = lambda flat, labels, rows, cols: _wide(flat[(  # noqa: E731
        _offsets(bat, labels, ext)[:, None, None] + _offsets(rows, labels, ext)[None, :, None]
        + _offsets(cols, labels, ext)[None, None, :])])
    prod = torch.matmul(grid(a, ia, m, k), grid(b, ib, k, n))
    c = torch.empty(_count(ic, ext), dtype=prod.dtype, device="cuda")
    at = (_offsets(bat, ic, ext)[:, None, None] + _offsets(m, ic, ext)[None, :, None]
          + _offsets(n, ic, ext)[None, None, :])
    c[at.reshape(-1)] = prod.reshape(-1)
    return c


def exact(case, seed):
    kind = case["kind"]
    if kind == "binary":
        ins, out, ext, flats = _operands(case, seed)
        c = _contract(flats[0], ins[0], flats[1], ins[1], out, ext)
        return c if case.get("inplace") else c.as_strided([ext[x] for x in out], _strides(out, ext))
    if kind == "hadamard":
        ins, out, ext, flats = _operands(case, seed)
        order = list(ins[0])
        return _wide(flats[0]) * _wide(flats[1])[_offsets(order, ins[1], ext)]
    if kind == "unary":
        ins, out, ext, flats = _operands(case, seed)
        summed = [x for x in dict.fromkeys(ins[0]) if x not in out]
        at = _offsets(list(out) + summed, ins[0], ext)
        return _wide(flats[0][at]).reshape(_count(summed, ext), _count(out, ext)).sum(0)
    if kind == "batch":
        pairs, offs = _batch_structure(case)
        pool = _batch_pool(case, seed)
        ext = dict.fromkeys({x for p in pairs for t in p for x in t}, 2)
        return torch.cat([_contract(pool[oa:], ia, pool[ob:], ib, ic, ext)
                          for (ia, ib, ic), (oa, ob) in zip(pairs, offs)])
    if kind == "svd":
        chi, d = case["chi"], case["d"]
        x = torch.randn(chi * d * d * chi, dtype=DTYPES[case["dtype"]], device="cuda", generator=_generator(seed))
        # the vectors are fixed only up to a phase each; the values are unique
        return [None, torch.linalg.svdvals(_wide(x).reshape(d * chi, chi * d).cpu()), None]
    specs, bank, leaves = _jobs(case, seed)
    roots = []
    for s, lv in zip(specs, leaves):
        labels = [list(x) for x in s.leaves] + [list(x[2]) for x in s.nodes]
        ext = dict.fromkeys({x for t in labels for x in t}, 2)
        vals = [t.parent().as_strided((1 << t.ndim,), (1,)) for t in lv]
        for a, b, o in s.nodes:
            vals.append(_contract(vals[a], labels[a], vals[b], labels[b], list(o), ext))
        roots.append(vals[-1])
    return roots
