// Contractions of power-of-two extents that do little work per output.
//
// A gate on a state vector, an outer-product-like pair of a circuit network
// (K <= 16) or one with a short output side does a few products per element of
// C it writes, so moving C and the operands bounds it.  With every extent a
// power of two, the offset of an element is the sum of its index bits'
// strides, and tiles can be cut from C in C's own address order whatever the
// order of its modes:
//   - a workgroup of 256 threads takes tiles of 2048 outputs; the 6 lowest
//     bits of C's address are the lane, so a store instruction writes 64
//     consecutive elements;
//   - the other tile bits (2 wave, 3 register bits) are chosen so that whole
//     128-byte lines of both operands belong to one tile and so that both
//     operands are reused (plan_bits);
//   - a tile's part of each operand is gathered in that operand's own address
//     order (per-thread constant offsets from a uniform base) and staged in
//     LDS with the lanes' bits lowest, folded so that neither the stores nor
//     the reads pile up on a bank; a K longer than fits is taken in chunks;
//   - each thread multiplies 2^r elements of the long operand by 2^(3-r) of the
//     short one, K after K in K's order;
//   - a workgroup runs several tiles, the next gather issued ahead of the
//     current tile's products and stores.
// Complex FP64, before (reduction, shallow or skinny kernel, tile GEMM) and now:
// a 2-qubit gate on 22 qubits (134 MB) 76.6 and 23.8 us (5.6 TB/s), on 24 341
// and 105; 2^12 x 2^12 x 2^2 86 and 76; 2^4 x 2^18 x 2^6 184 and 98; the
// shallow and skinny pairs of a 256-pair batch (8.2 GB) 3.2 and 2.1 ms.  Bound
// by memory; below some 100 tiles by fetching this code (8 KB a variant, run
// once) and the descriptor, so small contractions stay with the others, and by
// the round trip of every K chunk, so most with many chunks do (bits_for,
// bits_pays).  plan_bits leaves out what the tiles cannot hold: two long sides
// in C's default order, a tile over 4 GiB, an empty sum.
#include "bits.hpp"

#include <algorithm>

#include "device_types.hpp"
#include "kernels.hpp"

namespace mh {
namespace {

constexpr int NT = 1 << kBitThread;

typedef const MH_CONST BitDesc* DescPtr;  // read through the scalar cache

// The other vector-FMA kernels' sums in their order: a contraction's result does
// not depend on which of them runs it.
template <typename T, bool CP>
__device__ __forceinline__ void mac(Cplx<T>& acc, const Cplx<T>& a, const Cplx<T>& b) {
  acc.re = fma(a.re, b.re, acc.re);
  if constexpr (CP) {
    acc.re = fma(-a.im, b.im, acc.re);
    acc.im = fma(a.re, b.im, acc.im);
    acc.im = fma(a.im, b.re, acc.im);
  }
}

// Tiles [tile0, tile0 + d->run) of one contraction.  lds: the long operand's
// chunk, then the short one's.  LB: the long operand is the second one.
template <typename T, bool CP, int RL, bool LB>
__device__ __forceinline__ void bit_tiles(DescPtr d, uint32_t tile0, typename Elem<T, CP>::type* lds) {
  typedef typename Elem<T, CP>::type E;
  constexpr int RS = kBitReg - RL, FL = 1 << RL, FS = 1 << RS;
  constexpr uint32_t ES = sizeof(E);
  asm volatile("" ::"i"(RL * 2 + LB));  // keeps the variants apart (code hoisted out of their switch spilled)
  const uint32_t tid = threadIdx.x;
  // this thread's constant offsets (bytes)
  uint32_t tC = 0, tL = 0, tS = 0, gL = 0, gLl = 0, gS = 0, gSl = 0;
#pragma unroll
  for (int j = 0; j < kBitThread; ++j) {
    const uint32_t on = 0u - ((tid >> j) & 1u);
    tC += on & d->tC[j];
    tL ^= on & d->tL[j];
    tS ^= on & d->tS[j];
    gL += on & d->gL[j];
    gLl ^= on & d->gLl[j];
    gS += on & d->gS[j];
    gSl ^= on & d->gSl[j];
  }
  const int nl = d->nl, ns = d->ns;
  const bool in_l = (int)tid < nl, in_s = (int)tid < ns;
  E* const ldsS = lds + nl;
  uint32_t xl[FL], xs[FS];  // LDS elements read at k = 0
#pragma unroll
  for (int i = 0; i < FL; ++i) {
    xl[i] = tL;
#pragma unroll
    for (int b = 0; b < RL; ++b)
      if (i >> b & 1) xl[i] ^= d->rX[b];
  }
#pragma unroll
  for (int i = 0; i < FS; ++i) {
    xs[i] = tS;
#pragma unroll
    for (int b = 0; b < RS; ++b)
      if (i >> b & 1) xs[i] ^= d->rX[RL + b];
  }
  const uint32_t vL = gL * ES, vS = gS * ES, vC = tC * ES;
  uint32_t rC[kBitReg];
#pragma unroll
  for (int b = 0; b < kBitReg; ++b) rC[b] = d->rC[b];

  // offsets of tile0: lane j adds tile number bit j
  uint32_t oL = 0, oS = 0, oC = 0;
  {
    const int j = tid & 31;
    const MH_GLOBAL BitDesc* g = gptr<BitDesc>((const void*)d);
    if (tile0 >> j & 1) {
      oL = g->oL[j];
      oS = g->oS[j];
      oC = g->oC[j];
    }
#pragma unroll
    for (int m = 16; m; m >>= 1) {
      oL += __shfl_xor(oL, m, 64);
      oS += __shfl_xor(oS, m, 64);
      oC += __shfl_xor(oC, m, 64);
    }
    oL = __builtin_amdgcn_readfirstlane(oL);
    oS = __builtin_amdgcn_readfirstlane(oS);
    oC = __builtin_amdgcn_readfirstlane(oC);
  }
  const uint32_t tend = min(tile0 + (uint32_t)d->run, (uint32_t)d->tiles);
  const int nchunk = d->nchunk;
  Cplx<T> rl[kBitLongIt], rs[kBitShortIt];
  auto gather = [&](uint32_t ol, uint32_t os) {
    const char* const bl = (const char*)d->L + (uint64_t)ol * ES;
    const char* const bs = (const char*)d->S + (uint64_t)os * ES;
#pragma unroll
    for (int i = 0; i < kBitLongIt; ++i)
      if (i == 0 ? in_l : i * NT < nl) rl[i] = load_elem<T, CP>(bl + (uint64_t)d->iL[i] * ES + vL, 0);
#pragma unroll
    for (int i = 0; i < kBitShortIt; ++i)
      if (i == 0 ? in_s : i * NT < ns) rs[i] = load_elem<T, CP>(bs + (uint64_t)d->iS[i] * ES + vS, 0);
  };

  auto put = [](E& e, const Cplx<T>& v) {
    if constexpr (CP) {
      e.x = v.re;
      e.y = v.im;
    } else {
      e = v.re;
    }
  };
  gather(oL, oS);
  uint32_t kL = 0, kS = 0;  // offsets of the chunk gathered last
  Cplx<T> acc[FL][FS];
  for (uint32_t tile = tile0; tile < tend; ++tile) {
    for (int ch = 0; ch < nchunk; ++ch) {
      __syncthreads();  // the readers of the previous chunk are done
#pragma unroll
      for (int i = 0; i < kBitLongIt; ++i)
        if (i == 0 ? in_l : i * NT < nl) put(lds[gLl ^ d->iLl[i]], rl[i]);
#pragma unroll
      for (int i = 0; i < kBitShortIt; ++i)
        if (i == 0 ? in_s : i * NT < ns) put(ldsS[gSl ^ d->iSl[i]], rs[i]);
      __syncthreads();
      // the next chunk (or the next tile's first): a number's successor flips
      // its trailing ones, one entry of the step tables
      if (ch + 1 < nchunk) {
        const int j = __builtin_ctz(ch + 1);
        kL += d->cL[j];
        kS += d->cS[j];
        gather(oL + kL, oS + kS);
      } else if (tile + 1 < tend) {
        const int j = __builtin_ctz(tile + 1);
        oL += d->sL[j];
        oS += d->sS[j];
        kL = kS = 0;
        gather(oL, oS);
      }
      if (ch == 0) {
#pragma unroll
        for (int i = 0; i < FL; ++i)
#pragma unroll
          for (int j = 0; j < FS; ++j) acc[i][j] = Cplx<T>{T(0), T(0)};
      }
      const int kc = d->kc;
      const uint32_t sl = d->sl, ss = d->ss, kxl = d->kxl, kxs = d->kxs;
      for (int k = 0; k < kc; ++k) {
        Cplx<T> a[FL], b[FS];
#pragma unroll
        for (int i = 0; i < FL; ++i) {
          const E v = lds[(xl[i] ^ (k & kxl)) + k * sl];
          if constexpr (CP) a[i] = Cplx<T>{v.x, v.y};
          else a[i] = Cplx<T>{v, T(0)};
        }
#pragma unroll
        for (int j = 0; j < FS; ++j) {
          const E v = ldsS[(xs[j] ^ (k & kxs)) + k * ss];
          if constexpr (CP) b[j] = Cplx<T>{v.x, v.y};
          else b[j] = Cplx<T>{v, T(0)};
        }
#pragma unroll
        for (int i = 0; i < FL; ++i)
#pragma unroll
          for (int j = 0; j < FS; ++j) mac<T, CP>(acc[i][j], LB ? b[j] : a[i], LB ? a[i] : b[j]);
      }
    }
    char* const bc = (char*)d->C + (uint64_t)oC * ES;
    if (tile + 1 < tend) oC += d->sC[__builtin_ctz(tile + 1)];
    const bool nt = d->c_stream != 0;
#pragma unroll
    for (int i = 0; i < FL; ++i)
#pragma unroll
      for (int j = 0; j < FS; ++j) {
        uint32_t o = 0;
#pragma unroll
        for (int b = 0; b < RL; ++b)
          if (i >> b & 1) o += rC[b];
#pragma unroll
        for (int b = 0; b < RS; ++b)
          if (j >> b & 1) o += rC[RL + b];
        char* const p = bc + (uint64_t)o * ES + vC;
        if (nt) store_elem_nt<T, CP>(p, 0, acc[i][j]);
        else store_elem<T, CP>(p, 0, acc[i][j]);
      }
  }
}

template <typename T, bool CP>
__device__ __forceinline__ void bit_any(DescPtr d, uint32_t tile0, typename Elem<T, CP>::type* lds) {
  switch (d->reg_long * 2 + d->long_b) {
    case 2: bit_tiles<T, CP, 1, false>(d, tile0, lds); break;
    case 3: bit_tiles<T, CP, 1, true>(d, tile0, lds); break;
    case 4: bit_tiles<T, CP, 2, false>(d, tile0, lds); break;
    case 5: bit_tiles<T, CP, 2, true>(d, tile0, lds); break;
    case 6: bit_tiles<T, CP, 3, false>(d, tile0, lds); break;
    default: bit_tiles<T, CP, 3, true>(d, tile0, lds); break;
  }
}

template <typename T, bool CP>
__global__ __launch_bounds__(NT) void bits_kernel(BitArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  typename Elem<T, CP>::type* lds = reinterpret_cast<typename Elem<T, CP>::type*>(smem);
  const int2 w = a.items[blockIdx.x];
  bit_any<T, CP>((DescPtr)(a.descs + w.x), (uint32_t)w.y, lds);
}

// The descriptor travels in the kernel arguments: the plain call needs no table
// on the device.
template <typename T, bool CP>
__global__ __launch_bounds__(NT) void bits_one_kernel(BitDesc) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  typename Elem<T, CP>::type* lds = reinterpret_cast<typename Elem<T, CP>::type*>(smem);
#if defined(__HIP_DEVICE_COMPILE__)
  const DescPtr d = (DescPtr)__builtin_amdgcn_kernarg_segment_ptr();
  bit_any<T, CP>(d, blockIdx.x * (uint32_t)d->run, lds);
#endif
}

template <typename T, bool CP>
void one_t(const BitDesc& d, hipStream_t s) {
  const unsigned grid = (unsigned)((d.tiles + d.run - 1) / d.run);
  const size_t lds = (size_t)(d.nl + d.ns) * sizeof(typename Elem<T, CP>::type);
  hipLaunchKernelGGL((bits_one_kernel<T, CP>), dim3(grid), dim3(NT), lds, s, d);
}

}  // namespace

void launch_bits_one(bool dbl, bool cplx, const BitDesc& d, hipStream_t s) {
  if (dbl) {
    if (cplx) one_t<double, true>(d, s);
    else one_t<double, false>(d, s);
  } else {
    if (cplx) one_t<float, true>(d, s);
    else one_t<float, false>(d, s);
  }
}

void launch_bits(bool dbl, bool cplx, const BitArgs& a, int lds_elems, hipStream_t s) {
  if (a.nitems <= 0) return;
  const dim3 g((unsigned)a.nitems), b(NT);
  const size_t lds = (size_t)lds_elems * (dbl ? 8 : 4) * (cplx ? 2 : 1);
  if (dbl) {
    if (cplx) hipLaunchKernelGGL((bits_kernel<double, true>), g, b, lds, s, a);
    else hipLaunchKernelGGL((bits_kernel<double, false>), g, b, lds, s, a);
  } else {
    if (cplx) hipLaunchKernelGGL((bits_kernel<float, true>), g, b, lds, s, a);
    else hipLaunchKernelGGL((bits_kernel<float, false>), g, b, lds, s, a);
  }
}

}  // namespace mh
