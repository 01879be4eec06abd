// Host planning of the power-of-two kernel (bits.hip): which index bits a tile
// takes, and what each contributes to the offsets of C, of both operands and
// of their LDS copies.
#include "bits.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"

namespace mh {
namespace {

enum Cls { M = 0, N = 1, BATCH = 2 };

struct Bit {
  int cls;
  int64_t s[3];  // strides in A, B, C
};

// The bits of a dim list, fastest first; false unless every extent is a power
// of two (0, an empty sum, is none) and every stride is usable (nonnegative).
bool bits_of(const std::vector<Dim>& v, int cls, std::vector<Bit>& out) {
  for (auto& x : v) {
    if (x.extent < 1 || (x.extent & (x.extent - 1))) return false;
    for (int w = 0; w < 3; ++w)
      if (x.s[w] < 0) return false;
    for (int64_t e = 1; e < x.extent; e <<= 1) out.push_back(Bit{cls, {x.s[0] * e, x.s[1] * e, x.s[2] * e}});
  }
  return true;
}

// One bit of a gather: the operand's stride and the element's place in LDS.
struct Gather {
  int64_t stride;
  uint32_t lds;
};

// The gather's bits in the operand's address order: thread bits, then the
// iterations; returns the element count.
int plan_gather(std::vector<Gather> g, uint32_t* st, uint32_t* sl, uint32_t* it, uint32_t* il, int iterations) {
  std::stable_sort(g.begin(), g.end(), [](const Gather& x, const Gather& y) { return x.stride < y.stride; });
  for (int j = 0; j < kBitThread; ++j) {
    st[j] = j < (int)g.size() ? (uint32_t)g[(size_t)j].stride : 0;
    sl[j] = j < (int)g.size() ? g[(size_t)j].lds : 0;
  }
  for (int i = 0; i < iterations; ++i) {
    it[i] = il[i] = 0;
    for (size_t j = kBitThread; j < g.size(); ++j)
      if (i >> (j - kBitThread) & 1) {
        it[i] += (uint32_t)g[j].stride;
        il[i] ^= g[j].lds;
      }
  }
  return 1 << g.size();
}

}  // namespace

bool plan_bits(const ContractionDesc& d, BitDesc& out) {
  if (d.empty || !d.has_b || d.dt[0] != d.dt[2] || d.dt[1] != d.dt[2]) return false;
  const int64_t es = (int64_t)dtype_size(d.dt[2]);
  std::vector<Bit> c, k;
  if (!bits_of(d.m, M, c) || !bits_of(d.n, N, c) || !bits_of(d.batch, BATCH, c) || !bits_of(d.k, BATCH, k)) return false;
  const int nc = (int)c.size(), nk = (int)k.size();
  if (nc < kBitTile || nc - kBitTile > kBitOuter - 2 || nk > kBitChunk) return false;
  // every element offset fits 32 bits
  for (int w = 0; w < 3; ++w) {
    int64_t span = 1;
    for (auto& b : c) span += b.s[w];
    for (auto& b : k) span += b.s[w];
    if (span >= (int64_t(1) << 32)) return false;
  }
  std::stable_sort(c.begin(), c.end(), [](const Bit& x, const Bit& y) { return x.s[2] < y.s[2]; });
  if (c[0].s[2] == 0) return false;

  // The tile: the lane bits are C's lowest; then the bits along which a
  // 128-byte line of an operand runs (so that no other tile fetches the line
  // again); then C's next bits, from the class with fewer of them.
  std::vector<char> in((size_t)nc, 0);
  int taken = 0, count[3] = {0, 0, 0};
  auto take = [&](int i) {
    if (in[(size_t)i] || taken == kBitTile) return;
    in[(size_t)i] = 1;
    ++taken;
    ++count[c[(size_t)i].cls];
  };
  for (int i = 0; i < kBitLane; ++i) take(i);
  for (int64_t s = 1; s * es < 128; s <<= 1)
    for (int w = 0; w < 2; ++w)
      for (int i = 0; i < nc; ++i)
        if (c[(size_t)i].cls != (w == 0 ? N : M) && c[(size_t)i].s[w] == s) take(i);
  while (taken < kBitTile) {
    int best = -1;
    for (int i = 0; i < nc; ++i) {
      if (in[(size_t)i]) continue;
      const int x = c[(size_t)i].cls;
      auto rank = [&](int cls) { return cls == BATCH ? 64 : count[cls]; };
      if (best < 0 || rank(x) < rank(c[(size_t)best].cls)) best = i;
    }
    take(best);
  }
  const bool long_is_b = count[N] > count[M];
  const int lcls = long_is_b ? N : M, scls = long_is_b ? M : N, lw = long_is_b ? 1 : 0, sw = 1 - lw;
  const int lbits = count[lcls] + count[BATCH], sbits = count[scls] + count[BATCH];
  // K per chunk: both operands' elements within the kernel's gathers, and
  // within 2048 together where K is long (32 KB in complex FP64)
  const int lmax = kBitThread + 3, smax = kBitThread + 2;
  if (lbits > lmax || sbits > smax) return false;
  int kcb = std::min(nk, std::min(lmax - lbits, smax - sbits));
  while (kcb > 2 && (1 << (lbits + kcb)) + (1 << (sbits + kcb)) > 2048) --kcb;

  // Register bits: three of the tile's bits above the lanes, of M and N, two of
  // one and one of the other where there are; the other two are the wave's.
  std::vector<int> tile, lanes, upper;
  for (int i = 0; i < nc; ++i)
    if (in[(size_t)i]) (i < kBitLane ? lanes : upper).push_back(i);
  std::vector<int> ul, us, reg;
  for (int i : upper) {
    if (c[(size_t)i].cls == lcls) ul.push_back(i);
    if (c[(size_t)i].cls == scls) us.push_back(i);
  }
  const int rs = std::min<int>((int)us.size(), ul.size() >= 2 ? 1 : 2), rl = std::min<int>((int)ul.size(), kBitReg - rs);
  // (not taken: C's six lowest bits all of one side and more than five of the
  // other, such as the default output order where both sides are long; the
  // tile then has no upper bit of the long operand for a register)
  if (rl + rs != kBitReg || rl == 0) return false;
  reg.assign(ul.end() - rl, ul.end());
  reg.insert(reg.end(), us.end() - rs, us.end());
  std::vector<int> thread = lanes;
  for (int i : upper)
    if (std::find(reg.begin(), reg.end(), i) == reg.end()) thread.push_back(i);

  std::memset(&out, 0, sizeof out);
  out.reg_long = rl;
  out.long_b = long_is_b ? 1 : 0;
  // LDS places: per operand, its tile bits in thread, then register order;
  // bits past the banks' width are folded into the low ones
  const int fold = es == 16 ? 4 : es == 8 ? 5 : 6;
  int pl = 0, ps = 0;
  std::vector<uint32_t> place_l((size_t)nc, 0), place_s((size_t)nc, 0);
  auto mask = [&](int p) { return p < fold ? 1u << p : (1u << p) | 1u << ((p - fold) % fold); };
  auto place = [&](int i) {
    const int x = c[(size_t)i].cls;
    if (x != scls) place_l[(size_t)i] = mask(pl++);
    if (x != lcls) place_s[(size_t)i] = mask(ps++);
  };
  for (int i : thread) place(i);
  for (int i : reg) place(i);
  out.sl = 1 << lbits;
  out.ss = 1 << sbits;
  out.kxl = std::min(out.sl, 1 << fold) - 1;
  out.kxs = std::min(out.ss, 1 << fold) - 1;
  for (int j = 0; j < kBitThread; ++j) {
    const int i = thread[(size_t)j];
    out.tC[j] = (uint32_t)c[(size_t)i].s[2];
    out.tL[j] = place_l[(size_t)i];
    out.tS[j] = place_s[(size_t)i];
  }
  for (int j = 0; j < kBitReg; ++j) {
    const int i = reg[(size_t)j];
    out.rC[j] = (uint32_t)c[(size_t)i].s[2];
    out.rX[j] = j < rl ? place_l[(size_t)i] : place_s[(size_t)i];
  }
  // gathers
  std::vector<Gather> gl, gs;
  for (int i = 0; i < nc; ++i) {
    if (!in[(size_t)i]) continue;
    if (c[(size_t)i].cls != scls) gl.push_back(Gather{c[(size_t)i].s[lw], place_l[(size_t)i]});
    if (c[(size_t)i].cls != lcls) gs.push_back(Gather{c[(size_t)i].s[sw], place_s[(size_t)i]});
  }
  for (int j = 0; j < kcb; ++j) {
    gl.push_back(Gather{k[(size_t)j].s[lw], (uint32_t)(out.sl << j) | ((1u << j) & (uint32_t)out.kxl)});
    gs.push_back(Gather{k[(size_t)j].s[sw], (uint32_t)(out.ss << j) | ((1u << j) & (uint32_t)out.kxs)});
  }
  out.nl = plan_gather(gl, out.gL, out.gLl, out.iL, out.iLl, kBitLongIt);
  out.ns = plan_gather(gs, out.gS, out.gSl, out.iS, out.iSl, kBitShortIt);
  // a thread's own byte offsets are 32-bit registers: an operand that spreads a
  // tile over 4 GiB or more (a gate on a state of 2^30 ComplexF64 elements, its
  // new sites last) is left to the kernels with 64-bit offsets
  for (const uint32_t* s : {out.tC, out.gL, out.gS}) {
    uint64_t most = 0;
    for (int j = 0; j < kBitThread; ++j) most += s[j];
    if (most * (uint64_t)es >= uint64_t(1) << 32) return false;
  }
  out.kc = 1 << kcb;
  out.nchunk = 1 << (nk - kcb);
  for (int j = 0; j < nk; ++j)
    if (k[(size_t)j].s[lw] * es < 128) {
      ++out.line_k;
      if (j >= kcb) out.line_split = 1;
    }
  uint32_t cl = 0, cs = 0;  // the lower bits' strides together
  for (int j = kcb; j < nk; ++j) {
    const uint32_t x = (uint32_t)k[(size_t)j].s[lw], y = (uint32_t)k[(size_t)j].s[sw];
    out.cL[j - kcb] = x - cl;
    out.cS[j - kcb] = y - cs;
    cl += x;
    cs += y;
  }
  int o = 0;
  for (int i = 0; i < nc; ++i) {
    if (in[(size_t)i]) continue;
    out.oL[o] = (uint32_t)c[(size_t)i].s[lw];
    out.oS[o] = (uint32_t)c[(size_t)i].s[sw];
    out.oC[o] = (uint32_t)c[(size_t)i].s[2];
    ++o;
  }
  uint32_t sum[3] = {0, 0, 0};
  for (int j = 0; j < 4 && j < o; ++j) {
    out.sL[j] = out.oL[j] - sum[0];
    out.sS[j] = out.oS[j] - sum[1];
    out.sC[j] = out.oC[j] - sum[2];
    sum[0] += out.oL[j];
    sum[1] += out.oS[j];
    sum[2] += out.oC[j];
  }
  out.tiles = 1 << o;
  out.run = std::max(1, std::min(8, out.tiles / 2048));
  out.c_stream = es >= 16 && (double)(int64_t(1) << nc) * (double)es >= kStreamStoreBytes;
  return true;
}

}  // namespace mh
