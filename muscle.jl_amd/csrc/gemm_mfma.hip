// Gather-GEMM on CDNA4 matrix cores.
//
// C[bC + rowC[m] + colC[n]] = sum_k A[bA + rowA[m] + kA[k]] * B[bB + kB[k] + colB[n]]
//
// This replaces BackendBase's permutedims(a) / permutedims(b) / BLAS gemm /
// permutedims(c) sequence (src/Operations/binary_einsum.jl:89-95) with one
// kernel: operand tiles are gathered from their strided layout straight into
// LDS through per-mode offset tables, multiplied on MFMA, and scattered to C's
// own layout in the epilogue.
//
// Complex products run on real MFMAs either as 4M
//   re += ar*br - ai*bi,  im += ar*bi + ai*br               (4 MFMAs)
// or as 3M (Gauss):
//   P1 += ar*br, P2 += ai*bi, P3 += (ar+ai)*(br+bi);
//   re = P1 - P2, im = P3 - P1 - P2                         (3 MFMAs)
//
// One workgroup computes a BM x BN tile of C in K-tiles of BK, its waves
// arranged WM x WN, each wave a grid of MFMA 16x16x4 tiles.  Operands are
// staged in LDS as separate real and imaginary planes, double buffered, so one
// barrier per K-tile suffices; the gather of K-tile t + 1 is in flight while
// K-tile t is multiplied.
//
// What bounds the loop.  A vector instruction does not run beside an FP64 MFMA
// of the same SIMD: measured on the matrix cores alone, one VALU instruction
// between two FP64 MFMAs costs 12 cycles of matrix time (an MFMA takes 64), in
// a run of VALU instructions each further one 2.4 (32-bit) or 4.8 cycles
// (64-bit and FP64), whatever the number of waves; scalar instructions and LDS
// reads cost next to nothing.  So the loop keeps vector instructions out:
//   - a K-tile's elements are addressed from a wave-uniform base (the K offset
//     of the tile's first k, read through the scalar cache) plus one constant
//     32-bit register per element, wherever K's offsets split at multiples of
//     BK (SEP; the host checks it): no address arithmetic is left;
//   - LDS addresses are constant too (two K-tiles per loop pass, one per
//     buffer), and the tail of K is a step outside the loop, so no element is
//     checked inside it;
//   - the sums ar + ai and br + bi of the 3M form are taken in groups before a
//     run of MFMAs (scheduling barriers keep the compiler from spreading them).
// ComplexF64, M = N = K = 4096 on permuted layouts: 7.25 -> 5.64 ms (75.9 ->
// 97.5 TF, 93 % of the matrix cores' own rate for the 3M products); the loop
// before waited for each gather in front of its MFMAs and spent 1.8 vector
// instructions per MFMA.  ComplexF32 64 x 512^3: 574 -> 416 us (120 -> 165 TF).
// Real FP64 1497 x 1509 x 501: 85 -> 53 us.  Real FP64 4096^3 reaches 69 TF,
// real FP32 135 TF.  Without a common base per K-tile the ComplexF64 4096 cube
// takes 6.9 ms.
//
// Rows of BM + 16 elements put the four 16-lane groups of an MFMA operand read
// in disjoint LDS banks, and the column of element (k, m) is m ^ swz(k) (a
// permutation inside each aligned 16-block): the lanes that store consecutive
// k of one row (operands contiguous along K) then hit different banks.
// Workgroups are renumbered so each XCD (the dispatcher deals workgroups
// round-robin over 8 XCDs) gets a contiguous, grouped range of tiles and
// reuses A and B panels in its own L2.
//
// v_mfma_{f64_16x16x4f64, f32_16x16x4f32} lane layout on gfx950 (64 lanes),
// established with exact small-integer operands on the device:
//   A operand: lane l holds A[i = l % 16][k = l / 16]
//   B operand: lane l holds B[k = l / 16][j = l % 16]
//   D (4 regs), f32: lane l, reg r holds D[i = 4 * (l / 16) + r][j = l % 16]
//   D (4 regs), f64: lane l, reg r holds D[i = l / 16 + 4 * r][j = l % 16]
#include <algorithm>
#include <type_traits>

#include "device_types.hpp"
#include "kernels.hpp"

namespace mh {
namespace {

template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  static __device__ inline acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct Mfma<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  static __device__ inline acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int LDP = 16;  // LDS row padding (elements)

// LDS column of row (operand index) m at k: m ^ swz(k), a permutation inside
// each aligned 16-block.
template <typename T, int BK>
__device__ __forceinline__ constexpr int swz(int k) {
  if (BK == 16) return k & 15;
  return sizeof(T) == 8 ? (k & 6) << 1 : (k & 4) << 1;
}

// T: arithmetic type (MFMA precision); S: storage type of A, B and C.  S = T
// is the plain path; S = double with T = float is the FP32 rung of the
// precision ladder (operands rounded to FP32 as they are gathered).
// SEP: the offset of every k is that of its K-tile's first k plus that of its
// place in the tile, and a tile's elements span less than 2^32 bytes; else
// K offsets of every K-tile are looked up one K-tile ahead, into LDS.
// STEPS: MFMA steps (4 k each) whose operands are read and summed together.
template <typename T, typename S, bool CA, bool CB, bool G3, bool SEP, int BM, int BN, int BK, int WM, int WN, int OCC, int STEPS>
__global__ __launch_bounds__(64 * WM * WN, OCC) void gemm_tile_kernel(GemmArgs p) {
  using M_ = Mfma<T>;
  using acc_t = typename M_::acc_t;
  constexpr int NT = 64 * WM * WN;
  constexpr int NEA = BM * BK / NT, NEB = BN * BK / NT;
  constexpr int PA = CA ? 2 : 1, PB = CB ? 2 : 1;
  constexpr bool CC = CA || CB;
  constexpr int LA = BM + LDP, LB = BN + LDP;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16, KS = BK / 4;
  constexpr int SA = PA * BK * LA, SB = PB * BK * LB;  // elements of one stage
  constexpr int64_t EA = sizeof(S) * PA, EB = sizeof(S) * PB;
  static_assert(!G3 || (CA && CB), "3M needs two complex operands");
  static_assert(NEA >= 1 && NEB >= 1 && BM + BN <= NT, "tile shape");
  static_assert(2 * (SA + SB) * sizeof(T) >= (BM + BN) * sizeof(int64_t), "C's offsets reuse the stages");
  __shared__ __attribute__((aligned(16))) T lds[2 * (SA + SB)];  // two A stages, then two B stages

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  int tm, tn;
  gemm_tile_coords(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int bz = blockIdx.y;
  const int kbeg = blockIdx.z * p.kchunk;
  const int kend = min(p.K, kbeg + p.kchunk);
  const int nfull = (kend - kbeg) / BK, tail = (kend - kbeg) % BK;
  const bool to_partial = p.ksplit > 1;
  const bool AK = p.a_kmajor != 0, BKM = p.b_kmajor != 0;

  // this thread's element i of a K-tile: its k, its row (column)
  auto a_k = [&](int i) { return AK ? tid % BK : tid / BM + NT / BM * i; };
  auto b_k = [&](int i) { return BKM ? tid % BK : tid / BN + NT / BN * i; };
  auto a_m = [&](int i) { return AK ? tid / BK + NT / BK * i : tid % BM; };
  auto b_n = [&](int i) { return BKM ? tid / BK + NT / BK * i : tid % BN; };
  // Byte offsets in LDS, all constant: the stores of this thread's elements and
  // this lane's MFMA operand reads at step ks (row k = 4 ks + lane / 16, swizzled
  // column).  Kept opaque, each stays in a register of its own; buffers and
  // planes are a multiple of 64 elements apart, so a real and imaginary part
  // move in one instruction with immediate offsets.
  uint32_t wa[NEA], wb[NEB], xa[KS][TM], xb[KS][TN];
  auto opaque = [](uint32_t& v) { asm volatile("" : "+v"(v)); };
#pragma unroll
  for (int i = 0; i < NEA; ++i) {
    wa[i] = (uint32_t)sizeof(T) * (a_k(i) * LA + (a_m(i) ^ swz<T, BK>(a_k(i))));
    opaque(wa[i]);
  }
#pragma unroll
  for (int i = 0; i < NEB; ++i) {
    wb[i] = (uint32_t)sizeof(T) * (2 * SA + b_k(i) * LB + (b_n(i) ^ swz<T, BK>(b_k(i))));
    opaque(wb[i]);
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int kr = ks * 4 + (lane >> 4), c = (lane & 15) ^ swz<T, BK>(kr);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      xa[ks][i] = (uint32_t)sizeof(T) * (kr * LA + c + wm * (BM / WM) + i * 16);
      opaque(xa[ks][i]);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      xb[ks][j] = (uint32_t)sizeof(T) * (2 * SA + kr * LB + c + wn * (BN / WN) + j * 16);
      opaque(xb[ks][j]);
    }
  }
  auto at = [&](uint32_t off, int e) -> T& { return *((T*)((char*)lds + off) + e); };
  // not SEP: byte offsets in A (w = 0) and B of k of the K-tile in buffer b; in
  // FP64 in the padding of A's first rows (an array of its own left real FP64
  // 64x64x16 three workgroups per CU in place of four: 2048 x 2048 x 510 143 us
  // in place of 119)
  constexpr bool KPAD = sizeof(T) == 8;
  static_assert(BK <= LDP, "K offsets of one buffer and operand lie in one row's padding");
  __shared__ int64_t ktab[SEP || KPAD ? 1 : 4 * BK];
  auto koff = [&](int b, int w, int k) -> int64_t& {
    return KPAD ? ((int64_t*)lds)[(2 * b + w) * LA + BM + k] : ktab[(2 * b + w) * BK + k];
  };

  // K offsets of K-tile t (the last one's missing k clamped)
  auto k_offsets = [&](int t, int64_t* ka, int64_t* kb) {
    const int k0 = kbeg + t * BK, top = (t < nfull ? BK : tail) - 1;
    uint32_t ia[NEA], ib[NEB];
#pragma unroll
    for (int i = 0; i < NEA; ++i) ia[i] = (uint32_t)(k0 + min(a_k(i), top));
#pragma unroll
    for (int i = 0; i < NEB; ++i) ib[i] = (uint32_t)(k0 + min(b_k(i), top));
    load_offsets<NEA>(p.kA, ia, ka);
    load_offsets<NEB>(p.kB, ib, kb);
  };
  // Rows and columns outside M and N are clamped: they gather valid elements
  // whose products reach only outputs that are not stored.
  auto row_offsets = [&](int64_t* om, int64_t* on) {
    uint32_t im[NEA], in[NEB];
#pragma unroll
    for (int i = 0; i < NEA; ++i) im[i] = (uint32_t)min(m0 + a_m(i), p.M - 1);
#pragma unroll
    for (int i = 0; i < NEB; ++i) in[i] = (uint32_t)min(n0 + b_n(i), p.N - 1);
    load_offsets<NEA>(p.rowA, im, om);
    load_offsets<NEB>(p.colB, in, on);
  };
  // not SEP: K-tile t's entry of thread tid < 2 BK (A's k first, then B's)
  auto k_entry = [&](int t) {
    const uint32_t i[1] = {(uint32_t)min(kbeg + t * BK + tid % BK, kend - 1)};
    int64_t o[1];
    if (tid < BK) load_offsets<1>(p.kA, i, o);
    else load_offsets<1>(p.kB, i, o);
    return o[0] * (tid < BK ? EA : EB);
  };
  const int64_t offA0 = uniform_offset(p.bA, bz), offB0 = uniform_offset(p.bB, bz), offC0 = uniform_offset(p.bC, bz);
  Cplx<S> ra[NEA], rb[NEB];
  auto zero_tail = [&]() {  // both operands beyond K
#pragma unroll
    for (int i = 0; i < NEA; ++i)
      if (a_k(i) >= tail) ra[i] = Cplx<S>{S(0), S(0)};
#pragma unroll
    for (int i = 0; i < NEB; ++i)
      if (b_k(i) >= tail) rb[i] = Cplx<S>{S(0), S(0)};
  };
  const int nk = nfull + (tail ? 1 : 0);
  uint32_t va[NEA], vb[NEB];      // SEP: byte offsets inside a K-tile
  const char *pa[NEA], *pb[NEB];  // else: row (column) addresses
  const char* const bA = (const char*)p.A + (offA0 + p.minA) * EA;
  const char* const bB = (const char*)p.B + (offB0 + p.minB) * EB;
  {
    int64_t om[NEA], on[NEB], ka[NEA], kb[NEB];
    row_offsets(om, on);
    k_offsets(0, ka, kb);
#pragma unroll
    for (int i = 0; i < NEA; ++i) ra[i] = load_elem<S, CA>(p.A, offA0 + om[i] + ka[i]);
#pragma unroll
    for (int i = 0; i < NEB; ++i) rb[i] = load_elem<S, CB>(p.B, offB0 + on[i] + kb[i]);
    if constexpr (SEP) {
      const int64_t a0 = uniform_offset(p.kA, kbeg) + p.minA, b0 = uniform_offset(p.kB, kbeg) + p.minB;
#pragma unroll
      for (int i = 0; i < NEA; ++i) va[i] = (uint32_t)((om[i] + ka[i] - a0) * EA);
#pragma unroll
      for (int i = 0; i < NEB; ++i) vb[i] = (uint32_t)((on[i] + kb[i] - b0) * EB);
    } else {
#pragma unroll
      for (int i = 0; i < NEA; ++i) pa[i] = (const char*)p.A + (offA0 + om[i]) * EA;
#pragma unroll
      for (int i = 0; i < NEB; ++i) pb[i] = (const char*)p.B + (offB0 + on[i]) * EB;
      if (tid < 2 * BK && nk > 1) koff(1, tid / BK, tid % BK) = k_entry(1);
    }
    if (nfull == 0) zero_tail();
  }
  auto gather = [&](int t) {  // whole K-tile t (SEP), or any
    if constexpr (SEP) {
      const char* ga = bA + uniform_offset(p.kA, kbeg + t * BK) * EA;
      const char* gb = bB + uniform_offset(p.kB, kbeg + t * BK) * EB;
#pragma unroll
      for (int i = 0; i < NEA; ++i) {
        asm volatile("" : "+v"(va[i]));  // keeps the 32-bit offset a register of its own
        ra[i] = load_elem<S, CA>(ga + va[i], 0);
      }
#pragma unroll
      for (int i = 0; i < NEB; ++i) {
        asm volatile("" : "+v"(vb[i]));
        rb[i] = load_elem<S, CB>(gb + vb[i], 0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NEA; ++i) ra[i] = load_elem<S, CA>(pa[i] + koff(t & 1, 0, a_k(i)), 0);
#pragma unroll
      for (int i = 0; i < NEB; ++i) rb[i] = load_elem<S, CB>(pb[i] + koff(t & 1, 1, b_k(i)), 0);
    }
  };
  auto gather_tail = [&]() {  // the last K-tile, of fewer than BK k
    if constexpr (SEP) {
      int64_t om[NEA], on[NEB], ka[NEA], kb[NEB];
      row_offsets(om, on);
      k_offsets(nfull, ka, kb);
#pragma unroll
      for (int i = 0; i < NEA; ++i) ra[i] = load_elem<S, CA>(p.A, offA0 + om[i] + ka[i]);
#pragma unroll
      for (int i = 0; i < NEB; ++i) rb[i] = load_elem<S, CB>(p.B, offB0 + on[i] + kb[i]);
    } else {
      gather(nfull);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NEA; ++i) {
      at(wa[i], buf * SA) = (T)ra[i].re;
      if constexpr (CA) at(wa[i], buf * SA + BK * LA) = (T)ra[i].im;
    }
#pragma unroll
    for (int i = 0; i < NEB; ++i) {
      at(wb[i], buf * SB) = (T)rb[i].re;
      if constexpr (CB) at(wb[i], buf * SB + BK * LB) = (T)rb[i].im;
    }
  };

  acc_t acc0[TM][TN], acc1[TM][TN], acc2[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc0[i][j][r] = acc1[i][j][r] = acc2[i][j][r] = T(0);
  struct Frag {
    T ar[TM], ai[TM], as[TM], br[TN], bi[TN], bs[TN];
  };
  auto read_frag = [&](int buf, int ks, Frag& f) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      f.ar[i] = at(xa[ks][i], buf * SA);
      f.ai[i] = CA ? at(xa[ks][i], buf * SA + BK * LA) : T(0);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      f.br[j] = at(xb[ks][j], buf * SB);
      f.bi[j] = CB ? at(xb[ks][j], buf * SB + BK * LB) : T(0);
    }
  };
  auto sums = [&](Frag& f) {
    if constexpr (G3) {
#pragma unroll
      for (int i = 0; i < TM; ++i) f.as[i] = f.ar[i] + f.ai[i];
#pragma unroll
      for (int j = 0; j < TN; ++j) f.bs[j] = f.br[j] + f.bi[j];
    } else if constexpr (CA && CB) {
#pragma unroll
      for (int i = 0; i < TM; ++i) f.as[i] = -f.ai[i];
    }
  };
  auto multiply = [&](const Frag& f) {
    if constexpr (G3) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc0[i][j] = M_::mma(f.ar[i], f.br[j], acc0[i][j]);
          acc1[i][j] = M_::mma(f.ai[i], f.bi[j], acc1[i][j]);
          acc2[i][j] = M_::mma(f.as[i], f.bs[j], acc2[i][j]);
        }
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc0[i][j] = M_::mma(f.ar[i], f.br[j], acc0[i][j]);
          if constexpr (CB) acc1[i][j] = M_::mma(f.ar[i], f.bi[j], acc1[i][j]);
        }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (CA && CB) acc0[i][j] = M_::mma(f.as[i], f.bi[j], acc0[i][j]);
          if constexpr (CA) acc1[i][j] = M_::mma(f.ai[i], f.br[j], acc1[i][j]);
        }
    }
  };

  stash(0);
  __syncthreads();
  // K-tile t from LDS buffer cur; inner steps have a whole K-tile after theirs
  auto step = [&](int t, auto cur_, auto inner_) {
    constexpr int cur = decltype(cur_)::value;
    constexpr bool inner = decltype(inner_)::value;
    if (inner || t + 1 < nfull) gather(t + 1);
    else if (t + 1 < nk) gather_tail();
    int64_t kn = 0;  // K-tile t + 2's offsets replace K-tile t's
    if constexpr (!SEP)
      if (tid < 2 * BK && t + 2 < nk) kn = k_entry(t + 2);
    Frag f[STEPS];
#pragma unroll
    for (int k0 = 0; k0 < KS; k0 += STEPS) {
#pragma unroll
      for (int e = 0; e < STEPS; ++e) read_frag(cur, k0 + e, f[e]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < STEPS; ++e) sums(f[e]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < STEPS; ++e) multiply(f[e]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (inner || t + 1 < nk) {
      if (!inner && t + 1 == nfull) zero_tail();
      stash(cur ^ 1);
      if constexpr (!SEP)
        if (tid < 2 * BK && t + 2 < nk) koff(cur, tid / BK, tid % BK) = kn;
    }
    __syncthreads();
  };
  constexpr std::integral_constant<int, 0> B0;
  constexpr std::integral_constant<int, 1> B1;
  constexpr std::true_type inner;
  constexpr std::false_type ending;
  int t = 0;
  for (; t + 2 < nfull; t += 2) {
    step(t, B0, inner);
    step(t + 1, B1, inner);
  }
  step(t, B0, ending);
  if (t + 1 < nk) step(t + 1, B1, ending);
  if (t + 2 < nk) step(t + 2, B0, ending);

  // C's offsets, one lookup per thread, through the stages' LDS
  int64_t* coff = reinterpret_cast<int64_t*>(lds);
  if (!to_partial && tid < BM + BN) {
    const uint32_t i[1] = {(uint32_t)(tid < BM ? min(m0 + tid, p.M - 1) : min(n0 + tid - BM, p.N - 1))};
    int64_t o[1];
    if (tid < BM) load_offsets<1>(p.rowC, i, o);
    else load_offsets<1>(p.colC, i, o);
    coff[tid] = o[0];
  }
  __syncthreads();
  // partial sums of a split-K slice go to the workspace, [split][batch][m][n]
  const int64_t pbase = ((int64_t)blockIdx.z * gridDim.y + bz) * (int64_t)p.M * p.N;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int nl = wn * (BN / WN) + j * 16 + (lane & 15);
    if (n0 + nl >= p.N) continue;
    const int64_t cn = to_partial ? pbase + n0 + nl : offC0 + coff[BM + nl];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ml = wm * (BM / WM) + i * 16 + M_::row(lane, r);
        if (m0 + ml >= p.M) continue;
        T re, im;
        if constexpr (G3) {
          re = acc0[i][j][r] - acc1[i][j][r];
          im = acc2[i][j][r] - acc0[i][j][r] - acc1[i][j][r];
        } else {
          re = acc0[i][j][r];
          im = acc1[i][j][r];
        }
        if (to_partial) store_elem<T, CC>(p.partial, cn + (int64_t)(m0 + ml) * p.N, Cplx<T>{re, im});
        else if (p.c_stream) store_elem_nt<S, CC>(p.C, cn + coff[ml], Cplx<S>{(S)re, (S)im});
        else store_elem<S, CC>(p.C, cn + coff[ml], Cplx<S>{(S)re, (S)im});
      }
    }
  }
}
// C[bz, m, n] = sum over slices s of partial[s][bz][m][n], in slice order.
// Small (64-thread) workgroups spread the few outputs of a split-K GEMM over
// many CUs, and the unrolled slice loop keeps 8 loads of each thread in flight.
constexpr int NTF = 64;
template <typename T, typename S, bool CC>
__global__ __launch_bounds__(NTF) void splitk_finish_kernel(GemmArgs p) {
  const int64_t mn = (int64_t)p.M * p.N;
  const int64_t total = mn * p.batch;
  const int64_t o = (int64_t)blockIdx.x * NTF + threadIdx.x;
  if (o >= total) return;
  T re = 0, im = 0;
#pragma unroll 8
  for (int s = 0; s < p.ksplit; ++s) {
    const Cplx<T> v = load_elem<T, CC>(p.partial, (int64_t)s * total + o);
    re += v.re;
    im += v.im;
  }
  const int bz = (int)(o / mn);
  const int64_t r = o - bz * mn;
  const int m = (int)(r / p.N), n = (int)(r - (int64_t)m * p.N);
  store_elem<S, CC>(p.C, p.bC[bz] + p.rowC[m] + p.colC[n], Cplx<S>{(S)re, (S)im});
}

// A tile configuration of gemm_tile_kernel.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int OCC_, int STEPS_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, OCC = OCC_, STEPS = STEPS_;
};

// SEP: this kernel of the configuration (a common base per K-tile, or lookups).
template <typename T, typename S, bool CA, bool CB, bool G3, bool SEP, typename C>
void launch_kernel(GemmArgs g, hipStream_t s) {
  g.tiles_m = (g.M + C::BM - 1) / C::BM;
  g.tiles_n = (g.N + C::BN - 1) / C::BN;
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.batch, (unsigned)g.ksplit), block(64 * C::WM * C::WN);
  hipLaunchKernelGGL((gemm_tile_kernel<T, S, CA, CB, G3, SEP, C::BM, C::BN, C::BK, C::WM, C::WN, C::OCC, C::STEPS>), grid,
                     block, 0, s, g);
}
template <typename T, typename S, bool CA, bool CB, bool G3, typename C>
void launch_tile(const GemmArgs& g, hipStream_t s) {
  if (C::BK == 8 ? g.ktile8 : g.ktile16) launch_kernel<T, S, CA, CB, G3, true, C>(g, s);
  else launch_kernel<T, S, CA, CB, G3, false, C>(g, s);
}

// Tile shapes by the number of 64 x 64 tiles (and K slices) of the launch.
// Large tiles read the least; where there are too few of them to spread evenly
// over the workgroups that fit 256 CUs, smaller tiles win, and in complex FP64
// also where K is so short that a tile spends its time in its first loads and
// its stores.  Measured (us; N x N x 512 unless noted, tiles of 64 x 64 first):
//   complex FP64, 64x64x8 / 32x64x8 / 32x32x8: N = 1024: 80 / 66 / 58, 1536:
//     143 / 129 / 122, 2048: 231 / 203 / 213, 4096: 729 / 766 / 795;
//     4096 x 4096 with K = 8 / 32 / 128: 52 / 82 / 209 against 47 / 82 / 219
//     for 32x64x8; K = 4096: 5.69 ms, 5.59 with 64x64x16 (80 KB of LDS in place of
//     40, two workgroups per CU in place of three, half the barriers);
//   real FP64, 64x64x16 / 32x32x16: 1024: 32 / 26, 1536: 58 / 52, 2048: 75 / 88;
//   ComplexF32, 64x64x8 / 32x64x16: 1024: 46 / 34, 1536: 75 / 76, 2048: 101 / 110;
//   real FP32, 64x64x16 / 32x64x16: 1024: 22 / 17, 1536: 35 / 30, 2048: 43 / 49.
// K of at most 32 is one or two K-tiles, and a wave of stores per tile: real FP64
//   900 x 1900 x 16 8.8 / 10.0, 1200 x 2500 x 16 10.7 / 12.8, real FP32 the latter
//   9.0 / 10.6, ComplexF32 12.5 / 13.8; with a side below 64 and a last K-tile cut
//   off (looked up again) FP64 40000 x 2 x 24 10.8 / 7.9, FP32 131072 x 2 x 24 20.4 /
//   15.8, without FP32 65536 x 16 x 16 8.9 / 11.0.
// Where K's modes leave no common base per K-tile (lookups), a tile costs a
// chain of table reads before its first product:
//   slices of at most 64 k: 512 x 512 x 510 real FP64 22.8 / 27.5, FP32 16.9 / 22.1,
//     ComplexF32 25.7 / 29.5 (the FP32 rung's complex tiles 30.3 / 28.4), but real FP64 20 x
//     4000 x 500 22.5 / 19.4;
//   real FP64 from 640 tiles: 1900 x 1900 x 510 104 / 130;
//   three workgroups per CU take 768 tiles: ComplexF32 64x64x16 / 32x64x16 1024 x
//     3000 x 252 (768 tiles) 78 / 86, 1728 x 1728 x 1728 (729) 339 / 377, but 2048 x 2048
//     x 126 (1024) 73 / 65, 2197 x 2197 x 2197 710 / 801 (64x64x8 in its place); real x
//     complex FP64 2048 x 2048 x 126 78 / 73, 2300 x 2300 x 510 (1296) 245 / 260;
//     with K sliced ComplexF32 1000 x 1000 x 2197 187 / 162.
template <typename T, typename S, bool CA, bool CB, bool G3>
void launch_t(const GemmArgs& g, hipStream_t s) {
  const int64_t tiles = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64) * g.batch * g.ksplit;
  const int k = std::min(g.K, g.kchunk);
  const bool lookups = !((CA || CB) ? g.ktile8 : g.ktile16), wide = g.M >= 64 && g.N >= 64;
  const bool shortk = k <= 32 && wide, thin_tail = k <= 32 && !wide && g.K % 16;
  const bool brief = lookups && wide && g.ksplit > 1 && k <= 64 && tiles >= 256;
  if constexpr (sizeof(T) == 8 && CA && CB) {
    if (tiles < 1024) launch_tile<T, S, CA, CB, G3, Tile<32, 32, 8, 2, 2, 6, 1>>(g, s);
    else if (tiles < 2048 || k <= 32) launch_tile<T, S, CA, CB, G3, Tile<32, 64, 8, 2, 2, 4, 1>>(g, s);
    else if (G3 && k >= 1024 && g.ktile16) launch_kernel<T, S, CA, CB, G3, true, Tile<64, 64, 16, 2, 2, 2, 2>>(g, s);
    else launch_tile<T, S, CA, CB, G3, Tile<64, 64, 8, 2, 2, G3 ? 3 : 2, 1>>(g, s);
  } else if constexpr (sizeof(T) == 8) {
    if constexpr (CA || CB) {
      if (tiles < (lookups ? 1025 : 1024) && !brief) launch_tile<T, S, CA, CB, G3, Tile<32, 64, 8, 2, 2, 4, 2>>(g, s);
      else launch_tile<T, S, CA, CB, G3, Tile<64, 64, 8, 2, 2, 3, 1>>(g, s);
    } else {
      if (shortk ? tiles < 400 : thin_tail || (tiles < (lookups && wide ? 640 : 1024) && !brief)) launch_tile<T, S, CA, CB, G3, Tile<32, 32, 16, 2, 2, 6, 4>>(g, s);
      else launch_tile<T, S, CA, CB, G3, Tile<64, 64, 16, 2, 2, 4, 1>>(g, s);
    }
  } else if constexpr (CA || CB) {
    const bool whole = lookups && g.ksplit == 1;
    const bool small = whole ? tiles < 640 || (tiles > 768 && tiles <= 1024)
                             : tiles < (shortk ? 640 : lookups && sizeof(S) == 8 ? 1025 : 1024) && !(brief && sizeof(S) == 4);
    if (small) launch_tile<T, S, CA, CB, G3, Tile<32, 64, 16, 2, 2, 4, 1>>(g, s);
    else if (whole) launch_tile<T, S, CA, CB, G3, Tile<64, 64, 16, 2, 2, 3, 1>>(g, s);
    else launch_tile<T, S, CA, CB, G3, Tile<64, 64, 8, 2, 2, sizeof(S) == 8 ? 3 : 4, 1>>(g, s);
  } else {
    if (shortk ? tiles < 400 : thin_tail || (tiles < 1024 && !brief)) launch_tile<T, S, CA, CB, G3, Tile<32, 64, 16, 2, 2, 5, 4>>(g, s);
    else launch_tile<T, S, CA, CB, G3, Tile<64, 64, 16, 2, 2, sizeof(S) == 8 ? 3 : 4, 4>>(g, s);
  }
  if (g.ksplit > 1) {
    const int64_t total = (int64_t)g.M * g.N * g.batch;
    hipLaunchKernelGGL((splitk_finish_kernel<T, S, CA || CB>), dim3((unsigned)((total + NTF - 1) / NTF)), dim3(NTF),
                       0, s, g);
  }
}

}  // namespace

void launch_gemm_mfma(bool dbl, bool fp32_math, bool ca, bool cb, const GemmArgs& g0, hipStream_t s) {
  GemmArgs g = g0;
  if (g.ksplit < 1) {
    g.ksplit = 1;
    g.kchunk = g.K;
  }
  const bool g3 = ca && cb && g.complex3m;
  const int key = (dbl ? 8 : 0) | (ca ? 4 : 0) | (cb ? 2 : 0) | (g3 ? 1 : 0);
  if (dbl && fp32_math) {
    switch (key) {
      case 8: launch_t<float, double, false, false, false>(g, s); break;
      case 10: launch_t<float, double, false, true, false>(g, s); break;
      case 12: launch_t<float, double, true, false, false>(g, s); break;
      case 14: launch_t<float, double, true, true, false>(g, s); break;
      case 15: launch_t<float, double, true, true, true>(g, s); break;
    }
    return;
  }
  switch (key) {
    case 0: launch_t<float, float, false, false, false>(g, s); break;
    case 2: launch_t<float, float, false, true, false>(g, s); break;
    case 4: launch_t<float, float, true, false, false>(g, s); break;
    case 6: launch_t<float, float, true, true, false>(g, s); break;
    case 7: launch_t<float, float, true, true, true>(g, s); break;
    case 8: launch_t<double, double, false, false, false>(g, s); break;
    case 10: launch_t<double, double, false, true, false>(g, s); break;
    case 12: launch_t<double, double, true, false, false>(g, s); break;
    case 14: launch_t<double, double, true, true, false>(g, s); break;
    case 15: launch_t<double, double, true, true, true>(g, s); break;
  }
}

}  // namespace mh
