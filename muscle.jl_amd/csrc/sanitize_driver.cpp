// Host-side checks for the address/undefined-behaviour sanitizer build of the
// library's host code (lowering, planning, batch and server).  The driver is a
// plain executable, so the sanitizer runtime comes with it and nothing has to
// be preloaded into another process.
//
//   sanitize_driver          lowering and argument checking through
//                            muscle_hip_describe, and the tile GEMM's K-tile
//                            addressing against its offset tables (no GPU needed)
//   sanitize_driver --gpu    additionally: random contractions, a batch in all
//                            three run modes and a server with contraction-tree
//                            jobs, each against a naive host loop over every
//                            label assignment (einsum semantics: the output sums
//                            over the labels it does not carry)
//
// Exit status 0 when every check passed; the sanitizers abort on their own.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "batch.hpp"
#include "handle.hpp"
#include "muscle_hip.h"
#include "split.hpp"

namespace {

int g_failures = 0;

void expect(bool ok, const char* what, int64_t detail = 0) {
  if (ok) return;
  ++g_failures;
  std::fprintf(stderr, "FAIL: %s (%lld): %s\n", what, (long long)detail, muscle_hip_last_error());
}

// A tensor operand on the host: labels, extents and column-major strides of
// the listed order, possibly with gaps between elements.
struct Operand {
  std::vector<int32_t> modes;
  std::vector<int64_t> ext, strides;
  int64_t span = 1;  // elements from the first to one past the last
  muscle_hip_tensor_t desc(int dtype, void* data) const {
    muscle_hip_tensor_t t;
    t.dtype = dtype;
    t.rank = (int32_t)modes.size();
    t.data = data;
    t.modes = modes.data();
    t.extents = ext.data();
    t.strides = strides.data();
    return t;
  }
};

Operand make_operand(const std::vector<int32_t>& labels, const std::vector<int64_t>& extent, std::mt19937_64& rng) {
  Operand o;
  o.modes = labels;
  std::shuffle(o.modes.begin(), o.modes.end(), rng);
  int64_t s = 1 + (int64_t)(rng() % 2);  // a gap of one element now and then
  for (int32_t m : o.modes) {
    o.ext.push_back(extent[(size_t)m]);
    o.strides.push_back(s);
    s *= std::max<int64_t>(1, extent[(size_t)m]);
  }
  o.span = 1;
  for (size_t i = 0; i < o.modes.size(); ++i) o.span += (o.ext[i] - 1) * o.strides[i];
  if (o.span < 1) o.span = 1;
  return o;
}

// Roles of the labels of one contraction.
enum Role { BATCH, CONTRACT, LEFT, RIGHT, SUM_A, SUM_B, NROLES };

struct Case {
  std::vector<int64_t> extent;  // by label (label 0 unused)
  std::vector<int> role;
  Operand a, b, c;
};

Case random_case(std::mt19937_64& rng, int max_labels, int64_t max_ext, int64_t max_points) {
  Case cs;
  for (;;) {
    const int L = 1 + (int)(rng() % (uint64_t)max_labels);
    cs.extent.assign((size_t)L + 1, 1);
    cs.role.assign((size_t)L + 1, 0);
    std::vector<int32_t> la, lb, lc;
    int64_t points = 1;
    for (int l = 1; l <= L; ++l) {
      cs.extent[(size_t)l] = 1 + (int64_t)(rng() % (uint64_t)max_ext);
      const int r = (int)(rng() % 16);  // contracted and open labels are the common ones
      const int role = r < 4 ? CONTRACT : r < 8 ? LEFT : r < 12 ? RIGHT : r < 14 ? BATCH : r < 15 ? SUM_A : SUM_B;
      cs.role[(size_t)l] = role;
      points *= cs.extent[(size_t)l];
      if (role == BATCH || role == CONTRACT || role == LEFT || role == SUM_A) la.push_back(l);
      if (role == BATCH || role == CONTRACT || role == RIGHT || role == SUM_B) lb.push_back(l);
      if (role == BATCH || role == LEFT || role == RIGHT) lc.push_back(l);
    }
    if (points > max_points) continue;
    cs.a = make_operand(la, cs.extent, rng);
    cs.b = make_operand(lb, cs.extent, rng);
    cs.c = make_operand(lc, cs.extent, rng);
    // C must be dense (no gaps) so every element is written
    int64_t s = 1;
    for (size_t i = 0; i < cs.c.modes.size(); ++i) {
      cs.c.strides[i] = s;
      s *= std::max<int64_t>(1, cs.c.ext[i]);
    }
    cs.c.span = s;
    return cs;
  }
}

// ------------------------------------------------------------ no-GPU checks
void check_describe(std::mt19937_64& rng) {
  int checked = 0;
  for (int it = 0; it < 3000; ++it) {
    Case cs = random_case(rng, 9, 5, 1 << 22);
    const int precision = (int)(rng() % 5);
    const int dt = (int)(rng() % 4);  // MUSCLE_HIP_F32..C64
    muscle_hip_tensor_t c = cs.c.desc(dt, nullptr), a = cs.a.desc(dt, nullptr), b = cs.b.desc(dt, nullptr);
    muscle_hip_info_t info;
    int32_t modes[32], classes[32], nm = 0;
    const int st = muscle_hip_describe(&c, &a, &b, precision, 1e-10, &info, modes, classes, &nm);
    expect(st == MUSCLE_HIP_OK, "describe of a valid contraction", it);
    if (st != MUSCLE_HIP_OK) continue;
    // the fused extents multiply to the products of the label classes, times
    // those single-operand sums the plan folds into its K (the other operand
    // broadcast along them) instead of reducing them first
    int64_t pm = 1, pn = 1, pk = 1, pb = 1, ps = 1;
    for (size_t l = 1; l < cs.extent.size(); ++l) {
      const int r = cs.role[l];
      if (r == LEFT) pm *= cs.extent[l];
      if (r == RIGHT) pn *= cs.extent[l];
      if (r == CONTRACT) pk *= cs.extent[l];
      if (r == BATCH) pb *= cs.extent[l];
      if (r == SUM_A || r == SUM_B) ps *= cs.extent[l];
    }
    const int64_t base = pm * pn * pk * pb, fused = info.m * info.n * info.k * info.batch;
    expect(info.kernel == 0 || (fused % base == 0 && (base * ps) % fused == 0), "fused extents", it);
    // every label is classified as its role says (labels of extent 1 may merge away)
    for (int i = 0; i < nm; ++i) {
      const int l = modes[i];
      if (l <= 0 || l >= (int)cs.extent.size() || cs.extent[(size_t)l] == 1) continue;
      const int r = cs.role[(size_t)l];
      const int want_class = r == BATCH ? 0 : r == LEFT ? 1 : r == RIGHT ? 2 : r == CONTRACT ? 3 : r == SUM_A ? 4 : 5;
      expect(classes[i] == want_class, "label class", it * 100 + l);
    }
    ++checked;
  }
  // invalid inputs end in an error status, never in a crash
  Case cs = random_case(rng, 4, 3, 1 << 10);
  muscle_hip_tensor_t c = cs.c.desc(MUSCLE_HIP_C64, nullptr), a = cs.a.desc(MUSCLE_HIP_C64, nullptr),
                      b = cs.b.desc(MUSCLE_HIP_C64, nullptr);
  muscle_hip_info_t info;
  expect(muscle_hip_describe(nullptr, &a, &b, 0, 1e-10, &info, nullptr, nullptr, nullptr) != MUSCLE_HIP_OK,
         "null output descriptor");
  if (a.rank > 0) {
    std::vector<int64_t> bad(cs.a.ext);
    bad[0] += 1;
    muscle_hip_tensor_t a2 = a;
    a2.extents = bad.data();
    const bool shared = std::find(cs.b.modes.begin(), cs.b.modes.end(), cs.a.modes[0]) != cs.b.modes.end() ||
                        std::find(cs.c.modes.begin(), cs.c.modes.end(), cs.a.modes[0]) != cs.c.modes.end();
    if (shared)
      expect(muscle_hip_describe(&c, &a2, &b, 0, 1e-10, &info, nullptr, nullptr, nullptr) ==
                 MUSCLE_HIP_DIM_MISMATCH,
             "mismatched extents");
    std::vector<int64_t> neg(cs.a.ext);
    neg[0] = -3;
    a2.extents = neg.data();
    expect(muscle_hip_describe(&c, &a2, &b, 0, 1e-10, &info, nullptr, nullptr, nullptr) != MUSCLE_HIP_OK,
           "negative extent");
  }
  std::vector<int32_t> orphan(cs.c.modes);
  std::vector<int64_t> oext(cs.c.ext), ostr(cs.c.strides);
  orphan.push_back(999);
  oext.push_back(2);
  ostr.push_back(cs.c.span);
  muscle_hip_tensor_t c2 = c;
  c2.rank = (int32_t)orphan.size();
  c2.modes = orphan.data();
  c2.extents = oext.data();
  c2.strides = ostr.data();
  expect(muscle_hip_describe(&c2, &a, &b, 0, 1e-10, &info, nullptr, nullptr, nullptr) != MUSCLE_HIP_OK,
         "output label in neither operand");
  muscle_hip_tensor_t a3 = a;
  a3.dtype = 77;
  expect(muscle_hip_describe(&c, &a3, &b, 0, 1e-10, &info, nullptr, nullptr, nullptr) != MUSCLE_HIP_OK,
         "unknown dtype");
  expect(muscle_hip_describe(&c, &a, &b, 99, 1e-10, &info, nullptr, nullptr, nullptr) != MUSCLE_HIP_OK,
         "unknown precision");
  for (int s = 0; s < 9; ++s) expect(muscle_hip_status_string(s) != nullptr, "status string", s);
  for (int64_t m = 1; m < (int64_t(1) << 20); m *= 7) expect(muscle_hip_tuning_class(m, m + 3) >= 0, "size class", m);
  std::printf("describe: %d random contractions checked\n", checked);
}

// ------------------------------------------------------------ GPU checks
typedef std::complex<double> cd;

// Host values of an operand (as complex double) at its strided positions.
std::vector<cd> random_values(const Operand& o, std::mt19937_64& rng) {
  std::normal_distribution<double> nd;
  std::vector<cd> v((size_t)o.span);
  for (auto& x : v) x = cd(nd(rng), nd(rng));
  return v;
}

size_t esize(int dt) { return dt == MUSCLE_HIP_F32 ? 4 : dt == MUSCLE_HIP_F64 ? 8 : dt == MUSCLE_HIP_C32 ? 8 : 16; }
// A plan's K-tile addressing (ktile8, ktile16, min_a, min_b) against its offset
// tables: where a flag is set, off(k) = off(k - k mod bk) + off(k mod bk) for
// every k of both operands, and the elements of a K-tile lie in [min, min +
// 2^32 bytes).
void check_ktiles(std::mt19937_64& rng) {
  int64_t set = 0, plans = 0;
  for (int it = 0; it < 3000; ++it) {
    const int nk = 1 + (int)(rng() % 4);
    std::vector<int64_t> extent(1, 1);
    std::vector<int32_t> lk, la, lb, lc;
    for (int i = 0; i < nk; ++i) {
      const int64_t choices[] = {2, 2, 3, 4, 5, 8, 9, 16, 24, 33};
      extent.push_back(choices[rng() % 10]);
      lk.push_back((int32_t)extent.size() - 1);
    }
    extent.push_back(32 + (int64_t)(rng() % 40));
    la = lk;
    la.push_back((int32_t)extent.size() - 1);
    lc.push_back((int32_t)extent.size() - 1);
    extent.push_back(32 + (int64_t)(rng() % 40));
    lb = lk;
    lb.push_back((int32_t)extent.size() - 1);
    lc.push_back((int32_t)extent.size() - 1);
    Operand a = make_operand(la, extent, rng), b = make_operand(lb, extent, rng), c = make_operand(lc, extent, rng);
    for (auto& st : a.strides)
      if (rng() % 8 == 0) st = -st;  // reversed modes
    for (auto& st : b.strides)
      if (rng() % 64 == 0) st <<= 26;  // spans past 2^32 bytes
    const muscle_hip_tensor_t tc = c.desc(MUSCLE_HIP_F64, (void*)256), ta = a.desc(MUSCLE_HIP_F64, (void*)256),
                              tb = b.desc(MUSCLE_HIP_F64, (void*)256);
    const std::unique_ptr<mh::Plan> p =
        mh::build_contraction_plan(mh::lower_binary(tc, ta, tb), MUSCLE_HIP_PRECISION_NATIVE);
    if (p->kind != mh::Plan::GEMM) continue;
    ++plans;
    for (int64_t bk : {8, 16}) {
      bool splits = true, fits = true;
      for (int w = 0; w < 2; ++w) {
        const std::vector<int64_t> k = mh::offset_table(p->d.k, w), r = mh::offset_table(w == 0 ? p->d.m : p->d.n, w);
        for (size_t i = 0; i < k.size(); ++i)
          splits = splits && k[i] == k[i - i % (size_t)bk] + k[i % (size_t)bk];
        const int64_t lo = *std::min_element(r.begin(), r.end()), hi = *std::max_element(r.begin(), r.end());
        const size_t n = std::min<size_t>(k.size(), 16);
        const int64_t klo = *std::min_element(k.begin(), k.begin() + n), khi = *std::max_element(k.begin(), k.begin() + n);
        const int64_t base = w == 0 ? p->min_a : p->min_b;
        expect(base <= lo + klo, "K-tile base above an element", it);
        fits = fits && (hi + khi - base + 1) * 8 < (int64_t(1) << 32);
      }
      const bool flag = bk == 8 ? p->ktile8 : p->ktile16;
      expect(!flag || (splits && fits), "K-tile addressing of offsets that do not split or fit", it);
      set += flag;
    }
  }
  expect(set > plans / 2, "most plans have a common base per K-tile", set);
  std::printf("%lld tile GEMM plans checked, %lld K-tile sizes with a common base\n", (long long)plans, (long long)set);
}

// The FP32 rung's plan (FP64 operands rounded as they are gathered) has the
// addressing of the plain plan on the same operands.
void check_fp32_ktiles() {
  for (int64_t k : {48, 512, 1728})
    for (int dt : {MUSCLE_HIP_F64, MUSCLE_HIP_C64}) {
      Operand a{{1, 2}, {300, k}, {1, 300}}, b{{2, 3}, {k, 500}, {1, k}}, c{{1, 3}, {300, 500}, {1, 300}};
      const mh::ContractionDesc d = mh::lower_binary(c.desc(dt, (void*)256), a.desc(dt, (void*)256), b.desc(dt, (void*)256));
      const std::unique_ptr<mh::Plan> p = mh::build_contraction_plan(d, MUSCLE_HIP_PRECISION_NATIVE);
      const std::unique_ptr<mh::Plan> q = mh::build_contraction_plan(d, MUSCLE_HIP_PRECISION_FP32);
      mh::prepare_split(*q, 1e-6);
      expect(q->kind == mh::Plan::GEMM && q->fp32_math, "FP32 rung: plan", k);
      expect(p->ktile8 && p->ktile16 && q->ktile8 && q->ktile16, "FP32 rung: common base per K-tile", k);
      expect(p->min_a == q->min_a && p->min_b == q->min_b && p->gemm_kchunk == q->gemm_kchunk, "FP32 rung: base", k);
    }
}

// The power-of-two kernel's plan, run on the host index by index as the kernel
// does: every element lies inside its operand, the LDS copies are one-to-one,
// and C equals the naive sum over all labels, each output written once.
void check_bits(std::mt19937_64& rng) {
  int planned = 0, chunked = 0;
  for (int it = 0; it < 120; ++it) {
    std::vector<int64_t> extent(1, 1);
    std::vector<int32_t> la, lb, lc;
    auto label = [&](int64_t e) {
      extent.push_back(e);
      return (int32_t)extent.size() - 1;
    };
    // 11 to 14 output bits, mostly in modes of two, split unevenly over the
    // classes; 0 to 7 contracted bits
    int bits = 11 + (int)(rng() % 4), kbits = (int)(rng() % 8);
    const int pn = (int)(rng() % 11), nh = (int)(rng() % 3);
    for (int h = 0; h < nh; ++h) {
      const int32_t l = label(2);
      la.push_back(l);
      lb.push_back(l);
      lc.push_back(l);
    }
    bits -= nh;
    while (bits > 0) {
      const int w = std::min<int>(bits, rng() % 4 == 0 ? 3 : 1);
      const int32_t l = label(int64_t(1) << w);
      ((int)(rng() % 10) < pn ? lb : la).push_back(l);
      lc.push_back(l);
      bits -= w;
    }
    while (kbits > 0) {
      const int w = std::min<int>(kbits, rng() % 4 == 0 ? 2 : 1);
      const int32_t l = label(int64_t(1) << w);
      la.push_back(l);
      lb.push_back(l);
      kbits -= w;
    }
    Operand a = make_operand(la, extent, rng), b = make_operand(lb, extent, rng), c = make_operand(lc, extent, rng);
    const int dt = (int)(rng() % 4);
    const muscle_hip_tensor_t tc = c.desc(dt, (void*)256), ta = a.desc(dt, (void*)256), tb = b.desc(dt, (void*)256);
    const mh::ContractionDesc d = mh::lower_binary(tc, ta, tb);
    mh::BitDesc q;
    if (!mh::plan_bits(d, q)) continue;
    ++planned;
    chunked += q.nchunk > 1;
    q.run = std::min(q.tiles, 4);  // large launches run several tiles per workgroup
    // kernel operands (after the lowering's exchange)
    const Operand &A = d.swapped ? b : a, &B = d.swapped ? a : b;
    const Operand &L = q.long_b ? B : A, &S = q.long_b ? A : B;
    std::vector<int64_t> vl((size_t)L.span), vs((size_t)S.span), vc((size_t)c.span, 0), ref((size_t)c.span, 0);
    std::vector<char> seen((size_t)c.span, 0);
    for (auto& x : vl) x = (int64_t)(rng() % 201) - 100;
    for (auto& x : vs) x = (int64_t)(rng() % 201) - 100;
    const int FL = 1 << q.reg_long, FS = 1 << (mh::kBitReg - q.reg_long);
    auto bit_sum = [](uint32_t t, const uint32_t* s, int n) {
      uint32_t o = 0;
      for (int j = 0; j < n; ++j)
        if (t >> j & 1) o += s[j];
      return o;
    };
    auto bit_xor = [](uint32_t t, const uint32_t* s, int n) {
      uint32_t o = 0;
      for (int j = 0; j < n; ++j)
        if (t >> j & 1) o ^= s[j];
      return o;
    };
    bool inside = true, once = true, steps = true;
    const int NT = 1 << mh::kBitThread;
    for (uint32_t t0 = 0; t0 < (uint32_t)q.tiles; t0 += (uint32_t)q.run) {
      uint32_t oL = bit_sum(t0, q.oL, 32), oS = bit_sum(t0, q.oS, 32), oC = bit_sum(t0, q.oC, 32);
      for (uint32_t t = t0; t < t0 + (uint32_t)q.run; ++t) {
        std::vector<int64_t> acc((size_t)NT * 8, 0);
        uint32_t kL = 0, kS = 0;
        for (int ch = 0; ch < q.nchunk; ++ch) {
          std::vector<int64_t> ll((size_t)q.nl, 0), ls((size_t)q.ns, 0);
          std::vector<char> wl((size_t)q.nl, 0), ws((size_t)q.ns, 0);
          for (int tid = 0; tid < NT; ++tid) {
            for (int i = 0; i < mh::kBitLongIt; ++i) {
              if (!(i == 0 ? tid < q.nl : i * NT < q.nl)) continue;
              const uint64_t o = (uint64_t)(uint32_t)(oL + kL) + q.iL[i] + bit_sum((uint32_t)tid, q.gL, 8);
              const uint32_t x = bit_xor((uint32_t)tid, q.gLl, 8) ^ q.iLl[i];
              if (o >= vl.size() || x >= ll.size()) {
                inside = false;
                continue;
              }
              once = once && !wl[x];
              wl[x] = 1;
              ll[x] = vl[o];
            }
            for (int i = 0; i < mh::kBitShortIt; ++i) {
              if (!(i == 0 ? tid < q.ns : i * NT < q.ns)) continue;
              const uint64_t o = (uint64_t)(uint32_t)(oS + kS) + q.iS[i] + bit_sum((uint32_t)tid, q.gS, 8);
              const uint32_t x = bit_xor((uint32_t)tid, q.gSl, 8) ^ q.iSl[i];
              if (o >= vs.size() || x >= ls.size()) {
                inside = false;
                continue;
              }
              once = once && !ws[x];
              ws[x] = 1;
              ls[x] = vs[o];
            }
          }
          if (ch + 1 < q.nchunk) {
            kL += q.cL[__builtin_ctz(ch + 1)];
            kS += q.cS[__builtin_ctz(ch + 1)];
          }
          for (int tid = 0; tid < NT; ++tid)
            for (int i = 0; i < FL; ++i)
              for (int j = 0; j < FS; ++j)
                for (int k = 0; k < q.kc; ++k) {
                  const uint32_t x = ((bit_xor((uint32_t)tid, q.tL, 8) ^ bit_xor((uint32_t)i, q.rX, q.reg_long)) ^
                                      ((uint32_t)k & (uint32_t)q.kxl)) + (uint32_t)(k * q.sl);
                  const uint32_t y = ((bit_xor((uint32_t)tid, q.tS, 8) ^
                                       bit_xor((uint32_t)j, q.rX + q.reg_long, mh::kBitReg - q.reg_long)) ^
                                      ((uint32_t)k & (uint32_t)q.kxs)) + (uint32_t)(k * q.ss);
                  if (x >= ll.size() || y >= ls.size()) {
                    inside = false;
                    continue;
                  }
                  acc[(size_t)tid * 8 + (size_t)(i * FS + j)] += ll[x] * ls[y];
                }
        }
        for (int tid = 0; tid < NT; ++tid)
          for (int i = 0; i < FL; ++i)
            for (int j = 0; j < FS; ++j) {
              const uint64_t o = (uint64_t)oC + bit_sum((uint32_t)tid, q.tC, 8) + bit_sum((uint32_t)i, q.rC, q.reg_long) +
                                 bit_sum((uint32_t)j, q.rC + q.reg_long, mh::kBitReg - q.reg_long);
              if (o >= vc.size()) {
                inside = false;
                continue;
              }
              once = once && !seen[o];
              seen[o] = 1;
              vc[o] = acc[(size_t)tid * 8 + (size_t)(i * FS + j)];
            }
        if (t + 1 < t0 + (uint32_t)q.run) {
          const int j = __builtin_ctz(t + 1);
          oL += q.sL[j];
          oS += q.sS[j];
          oC += q.sC[j];
          steps = steps && oL == bit_sum(t + 1, q.oL, 32) && oS == bit_sum(t + 1, q.oS, 32) &&
                  oC == bit_sum(t + 1, q.oC, 32);
        }
      }
    }
    expect(inside, "power-of-two plan: an index outside its buffer", it);
    expect(once, "power-of-two plan: an element written twice", it);
    expect(steps, "power-of-two plan: tile steps", it);
    // naive sum over all label assignments
    std::vector<int64_t> idx(extent.size(), 0);
    auto off = [&](const Operand& o) {
      int64_t r = 0;
      for (size_t i = 0; i < o.modes.size(); ++i) r += idx[(size_t)o.modes[i]] * o.strides[i];
      return (size_t)r;
    };
    for (;;) {
      ref[off(c)] += vl[off(L)] * vs[off(S)];
      size_t l = 1;
      while (l < extent.size() && ++idx[l] == extent[l]) idx[l++] = 0;
      if (l == extent.size()) break;
    }
    expect(vc == ref, "power-of-two plan: result", it);
  }
  expect(planned > 80 && chunked > 10, "power-of-two plans", planned);
  std::printf("power-of-two kernel: %d plans run on the host, %d with K chunks\n", planned, chunked);
}

// Operands too large to hold here, by their strides alone: wherever the
// power-of-two kernel takes a contraction, the byte offsets that its threads
// form in 32 bits have the value they have in 64, and its steps from tile to
// tile land where the tile's number says.
void check_bits_offsets(std::mt19937_64& rng) {
  int planned = 0, large = 0;
  auto check = [&](const muscle_hip_tensor_t& tc, const muscle_hip_tensor_t& ta, const muscle_hip_tensor_t& tb,
                   int64_t detail) {
    mh::BitDesc q;
    const mh::ContractionDesc d = mh::lower_binary(tc, ta, tb);
    if (!mh::plan_bits(d, q)) return false;
    ++planned;
    const uint32_t ES = (uint32_t)esize(tc.dtype);
    bool same = true, steps = true;
    for (uint32_t tid = 0; tid < (1u << mh::kBitThread); ++tid)
      for (const uint32_t* s : {q.tC, q.gL, q.gS}) {
        uint32_t v = 0;
        uint64_t exact = 0;
        for (int j = 0; j < mh::kBitThread; ++j)
          if (tid >> j & 1) {
            v += s[j];
            exact += s[j];
          }
        same = same && (uint64_t)(uint32_t)(v * ES) == exact * ES;
      }
    const uint32_t* o[3] = {q.oL, q.oS, q.oC};
    const uint32_t* st[3] = {q.sL, q.sS, q.sC};
    for (int w = 0; w < 3; ++w) {
      auto at = [&](uint32_t t) {
        uint32_t x = 0;
        for (int j = 0; j < mh::kBitOuter; ++j)
          if (t >> j & 1) x += o[w][j];
        return x;
      };
      for (uint32_t t0 : {0u, (uint32_t)(q.tiles - q.run)})
        for (uint32_t t = t0; t + 1 < t0 + (uint32_t)q.run; ++t)
          steps = steps && at(t) + st[w][__builtin_ctz(t + 1)] == at(t + 1);
    }
    large += q.run == 8;
    expect(same, "power-of-two plan: a thread's byte offset beyond 32 bits", detail);
    expect(steps, "power-of-two plan: tile steps of a full run", detail);
    return true;
  };
  // gates on states of up to 2^32 elements, the new sites last in the output
  for (int dt = 0; dt < 4; ++dt)
    for (int sites = 26; sites <= 32; ++sites)
      for (int it = 0; it < 24; ++it) {
        const int qubits = 1 + it % 3;
        std::vector<int32_t> all((size_t)sites);
        for (int i = 0; i < sites; ++i) all[(size_t)i] = i + 1;
        std::shuffle(all.begin(), all.end(), rng);
        Operand st, g, c;
        auto mode = [&](Operand& x, int32_t l) {
          x.modes.push_back(l);
          x.ext.push_back(2);
          x.strides.push_back(int64_t(1) << (x.modes.size() - 1));
        };
        for (int l = 1; l <= sites; ++l) {
          mode(st, l);
          if (std::find(all.begin(), all.begin() + qubits, l) == all.begin() + qubits) mode(c, l);
        }
        for (int i = 0; i < qubits; ++i) mode(g, sites + 1 + i);
        for (int i = 0; i < qubits; ++i) mode(g, all[(size_t)i]);
        for (int i = 0; i < qubits; ++i) mode(c, sites + 1 + i);
        const bool ok = check(c.desc(dt, (void*)256), st.desc(dt, (void*)256), g.desc(dt, (void*)256), sites * 100 + it);
        expect(ok || sites >= 29 || qubits == 1, "a gate on a state of 2 to 4 GB stays with the power-of-two kernel",
               sites * 100 + it);
      }
  // strided views: a wide gap above one mode of one operand
  for (int it = 0; it < 600; ++it) {
    std::vector<int64_t> extent(1, 1);
    std::vector<int32_t> la, lb, lc;
    const int bits = 11 + (int)(rng() % 4), kbits = 1 + (int)(rng() % 4);
    for (int i = 0; i < bits + kbits; ++i) {
      extent.push_back(2);
      const int32_t l = (int32_t)extent.size() - 1;
      if (i < bits) lc.push_back(l);
      const int to = (int)(rng() % 2);
      if (i >= bits || to == 0) la.push_back(l);
      if (i >= bits || to == 1) lb.push_back(l);
    }
    Operand x[3] = {make_operand(la, extent, rng), make_operand(lb, extent, rng), make_operand(lc, extent, rng)};
    Operand& y = x[rng() % 3];
    if (y.strides.empty()) continue;
    const size_t from = rng() % y.strides.size();
    const int shift = 10 + (int)(rng() % 14);
    for (size_t i = from; i < y.strides.size(); ++i) y.strides[i] <<= shift;
    const int dt = (int)(rng() % 4);
    check(x[2].desc(dt, (void*)256), x[0].desc(dt, (void*)256), x[1].desc(dt, (void*)256), it);
  }
  expect(planned > 300 && large > 100, "power-of-two plans of large operands", planned);
  std::printf("power-of-two kernel: offsets of %d plans of large operands checked\n", planned);
}

// A contracted mode without elements (M = 2^16, N = 4 and M = 2^18, N = 1 are
// large enough for the power-of-two kernel otherwise): the sum is empty, and
// neither operand has an element to read.
void check_bits_empty() {
  int others = 0;
  for (int dt = 0; dt < 4; ++dt)
    for (int64_t n : {1, 4})
      for (int64_t k2 : {1, 2})
        for (int64_t k : {0, 2}) {
          const int64_t m = n == 1 ? 1 << 18 : 1 << 16;
          Operand a{{1, 3, 4}, {m, k, k2}, {1, m, m * 2}}, b{{3, 4, 2}, {k, k2, n}, {1, 2, 2 * k2}},
              c{{1, 2}, {m, n}, {1, m}};
          const muscle_hip_tensor_t tc = c.desc(dt, (void*)256), ta = a.desc(dt, k ? (void*)256 : nullptr),
                                    tb = b.desc(dt, k ? (void*)256 : nullptr);
          const mh::ContractionDesc d = mh::lower_binary(tc, ta, tb);
          mh::BitDesc q;
          const int kind = mh::build_contraction_plan(d, MUSCLE_HIP_PRECISION_NATIVE)->kind;
          if (k == 0) {
            expect(!mh::plan_bits(d, q), "power-of-two plan of an empty sum", dt * 100 + n * 10 + k2);
            expect(kind == mh::Plan::REDUCE, "kernel of an empty sum", kind);
          } else if (kind == mh::Plan::BITS) {
            ++others;
          }
        }
  expect(others > 0, "the same sizes with elements to sum", others);
}

// Which contractions the power-of-two kernel takes, plain and in a batch, on
// both sides of the rules' lines: sides of 2^s and 2^n, K of 2^k, modes of two.
// The long operand's lines run along its rows, or along K (kfast), or along
// both (half of a line each); C has the short side's modes first.
void check_bits_rules() {
  enum Lines { ROWS, KFAST, HALF };
  const int F32 = MUSCLE_HIP_F32, F64 = MUSCLE_HIP_F64, C32 = MUSCLE_HIP_C32, C64 = MUSCLE_HIP_C64;
  struct {
    int dt, s, n, k;
    Lines lines;
    bool plain, batch;
  } rows[] = {
      // one and two chunks, by tiles
      {C64, 4, 14, 2, ROWS, true, false}, {C64, 4, 13, 2, ROWS, false, false}, {C64, 4, 15, 2, ROWS, true, true},
      {F32, 3, 15, 3, ROWS, false, false}, {F32, 3, 16, 3, ROWS, true, true}, {F64, 2, 17, 4, ROWS, false, true},
      // a short side and K in many chunks
      {C64, 2, 18, 7, ROWS, true, false}, {C64, 2, 18, 7, KFAST, true, true}, {C64, 1, 19, 6, KFAST, false, false},
      {C64, 0, 18, 3, HALF, false, false}, {C64, 0, 20, 3, ROWS, true, false}, {C64, 4, 16, 7, ROWS, true, true},
      {F64, 2, 18, 7, ROWS, true, false}, {F64, 2, 18, 7, HALF, false, false}, {F64, 2, 18, 7, KFAST, true, true},
      {F64, 0, 20, 3, HALF, false, false}, {F64, 0, 20, 3, KFAST, false, false}, {F64, 4, 16, 7, ROWS, false, false},
      {C32, 1, 19, 5, KFAST, false, true}, {C32, 3, 17, 6, HALF, false, false}, {C32, 3, 18, 6, HALF, true, false},
      {F32, 3, 18, 6, HALF, false, false}, {F32, 4, 16, 5, ROWS, false, false}, {F32, 4, 16, 6, KFAST, false, true},
      {F32, 1, 19, 5, ROWS, true, false}, {F32, 1, 19, 5, HALF, false, false},
      // K beyond 128, both sides long
      {C64, 3, 17, 8, KFAST, false, false}, {C64, 5, 15, 5, ROWS, false, false}, {C64, 5, 6, 3, ROWS, true, false},
      {F32, 5, 15, 4, ROWS, true, true}, {F64, 5, 17, 4, ROWS, false, true},
  };
  mh::Handle h;
  int i = 0;
  for (const auto& r : rows) {
    Operand a, b, c;
    auto put = [](Operand& o, int from, int count) {
      for (int j = 0; j < count; ++j) {
        o.strides.push_back(int64_t(1) << o.modes.size());
        o.modes.push_back(from + j);
        o.ext.push_back(2);
      }
    };
    const int S = 1, N = S + r.s, K = N + r.n;
    int line = 0;  // log2 of the elements of a line
    while ((int64_t)esize(r.dt) << line < 128) ++line;
    put(a, S, r.s);
    put(a, K, r.k);
    const int first = r.lines == ROWS ? 0 : r.lines == KFAST ? r.k : std::min(r.k, line - 1);
    put(b, K, first);
    put(b, N, r.n);
    put(b, K + first, r.k - first);
    put(c, S, r.s);
    put(c, N, r.n);
    const mh::ContractionDesc d =
        mh::lower_binary(c.desc(r.dt, (void*)256), a.desc(r.dt, (void*)256), b.desc(r.dt, (void*)256));
    mh::BitDesc q;
    expect(mh::plan_bits(d, q), "power-of-two rule: the kernel could take it", i);
    const bool plain = mh::build_contraction_plan(d, MUSCLE_HIP_PRECISION_NATIVE)->kind == mh::Plan::BITS;
    mh::PlannedPair pair;
    std::vector<int64_t> tab;
    pair.d = d;
    mh::plan_pair(h, pair, tab, MUSCLE_HIP_TILE_AUTO, mh::kTickSingleMax);
    if (plain != r.plain || pair.bits != r.batch)
      std::fprintf(stderr, "row %d: %d chunks, %d K bits in a line, %d tiles: plain %d, batch %d\n", i, q.nchunk, q.line_k,
                   q.tiles, plain, pair.bits);
    expect(plain == r.plain, "power-of-two rule: plain contraction", i);
    expect(pair.bits == r.batch, "power-of-two rule: batched pair", i);
    ++i;
  }
  std::printf("power-of-two kernel: %d contractions on both sides of its rules\n", i);
}

bool is_cplx(int dt) { return dt == MUSCLE_HIP_C32 || dt == MUSCLE_HIP_C64; }

std::vector<char> encode(const std::vector<cd>& v, int dt) {
  std::vector<char> out(v.size() * esize(dt));
  for (size_t i = 0; i < v.size(); ++i) {
    switch (dt) {
      case MUSCLE_HIP_F32: reinterpret_cast<float*>(out.data())[i] = (float)v[i].real(); break;
      case MUSCLE_HIP_F64: reinterpret_cast<double*>(out.data())[i] = v[i].real(); break;
      case MUSCLE_HIP_C32:
        reinterpret_cast<float*>(out.data())[2 * i] = (float)v[i].real();
        reinterpret_cast<float*>(out.data())[2 * i + 1] = (float)v[i].imag();
        break;
      default:
        reinterpret_cast<double*>(out.data())[2 * i] = v[i].real();
        reinterpret_cast<double*>(out.data())[2 * i + 1] = v[i].imag();
    }
  }
  return out;
}

cd decode(const std::vector<char>& buf, int dt, size_t i) {
  switch (dt) {
    case MUSCLE_HIP_F32: return cd(reinterpret_cast<const float*>(buf.data())[i], 0.0);
    case MUSCLE_HIP_F64: return cd(reinterpret_cast<const double*>(buf.data())[i], 0.0);
    case MUSCLE_HIP_C32:
      return cd(reinterpret_cast<const float*>(buf.data())[2 * i], reinterpret_cast<const float*>(buf.data())[2 * i + 1]);
    default:
      return cd(reinterpret_cast<const double*>(buf.data())[2 * i], reinterpret_cast<const double*>(buf.data())[2 * i + 1]);
  }
}

// C[c] = sum over the labels C lacks of A[a] B[b], every label assignment visited once.
std::vector<cd> reference(const Case& cs, const std::vector<cd>& A, const std::vector<cd>& B, bool cplx) {
  const size_t L = cs.extent.size() - 1;
  std::vector<cd> C((size_t)cs.c.span, cd(0, 0));
  std::vector<int64_t> idx(L + 1, 0);
  auto offset = [&](const Operand& o) {
    int64_t off = 0;
    for (size_t i = 0; i < o.modes.size(); ++i) off += idx[(size_t)o.modes[i]] * o.strides[i];
    return off;
  };
  for (int64_t e : cs.extent)
    if (e == 0) return C;
  for (;;) {
    cd x = A[(size_t)offset(cs.a)], y = B[(size_t)offset(cs.b)];
    if (!cplx) {
      x = cd(x.real(), 0);
      y = cd(y.real(), 0);
    }
    C[(size_t)offset(cs.c)] += x * y;
    size_t l = 1;
    for (; l <= L; ++l) {
      if (++idx[l] < cs.extent[l]) break;
      idx[l] = 0;
    }
    if (l > L) break;
  }
  return C;
}

double rel_err(const std::vector<cd>& got, const std::vector<cd>& want) {
  double num = 0, den = 0;
  for (size_t i = 0; i < got.size(); ++i) {
    num += std::norm(got[i] - want[i]);
    den += std::norm(want[i]);
  }
  return den > 0 ? std::sqrt(num / den) : std::sqrt(num);
}

struct DevCase {
  Case cs;
  int dt;
  std::vector<cd> A, B, want;
  void *da = nullptr, *db = nullptr, *dc = nullptr;
  muscle_hip_tensor_t ta, tb, tc;
};

DevCase make_dev_case(std::mt19937_64& rng, int dt) {
  DevCase d;
  d.cs = random_case(rng, 7, 6, 1 << 16);
  d.dt = dt;
  d.A = random_values(d.cs.a, rng);
  d.B = random_values(d.cs.b, rng);
  d.want = reference(d.cs, d.A, d.B, is_cplx(dt));
  const auto ha = encode(d.A, dt), hb = encode(d.B, dt);
  expect(hipMalloc(&d.da, ha.size()) == hipSuccess && hipMalloc(&d.db, hb.size()) == hipSuccess &&
             hipMalloc(&d.dc, (size_t)d.cs.c.span * esize(dt)) == hipSuccess,
         "hipMalloc");
  expect(hipMemcpy(d.da, ha.data(), ha.size(), hipMemcpyHostToDevice) == hipSuccess, "copy A");
  expect(hipMemcpy(d.db, hb.data(), hb.size(), hipMemcpyHostToDevice) == hipSuccess, "copy B");
  expect(hipMemset(d.dc, 0x7f, (size_t)d.cs.c.span * esize(dt)) == hipSuccess, "poison C");
  d.ta = d.cs.a.desc(dt, d.da);
  d.tb = d.cs.b.desc(dt, d.db);
  d.tc = d.cs.c.desc(dt, d.dc);
  return d;
}

double dev_error(const DevCase& d) {
  std::vector<char> buf((size_t)d.cs.c.span * esize(d.dt));
  expect(hipMemcpy(buf.data(), d.dc, buf.size(), hipMemcpyDeviceToHost) == hipSuccess, "copy C");
  std::vector<cd> got(d.want.size());
  for (size_t i = 0; i < got.size(); ++i) got[i] = decode(buf, d.dt, i);
  return rel_err(got, d.want);
}

void free_dev_case(DevCase& d) {
  expect(hipFree(d.da) == hipSuccess && hipFree(d.db) == hipSuccess && hipFree(d.dc) == hipSuccess, "hipFree");
}

double tolerance(int dt) { return dt == MUSCLE_HIP_F32 || dt == MUSCLE_HIP_C32 ? 2e-5 : 1e-12; }

void check_gpu(std::mt19937_64& rng) {
  muscle_hip_handle_t h = nullptr;
  expect(muscle_hip_create(&h) == MUSCLE_HIP_OK, "create handle");
  if (!h) return;
  // single contractions, every dtype
  int n_single = 0;
  for (int it = 0; it < 80; ++it) {
    const int dt = (int)(rng() % 4);
    DevCase d = make_dev_case(rng, dt);
    muscle_hip_info_t info;
    const int st = muscle_hip_binary_einsum(h, &d.tc, &d.ta, &d.tb, 0, 1e-12, &info);
    expect(st == MUSCLE_HIP_OK, "binary_einsum", it);
    expect(muscle_hip_synchronize(h) == MUSCLE_HIP_OK, "synchronize", it);
    if (st == MUSCLE_HIP_OK) {
      const double e = dev_error(d);
      expect(e <= tolerance(dt), "binary_einsum result", it);
      ++n_single;
    }
    free_dev_case(d);
  }
  // one batch of ComplexF64 pairs, in every run mode
  std::vector<DevCase> pairs;
  for (int i = 0; i < 40; ++i) pairs.push_back(make_dev_case(rng, MUSCLE_HIP_C64));
  std::vector<muscle_hip_tensor_t> cs, as, bs;
  for (auto& d : pairs) {
    cs.push_back(d.tc);
    as.push_back(d.ta);
    bs.push_back(d.tb);
  }
  muscle_hip_batch_t batch = nullptr;
  expect(muscle_hip_batch_create(h, (int64_t)pairs.size(), cs.data(), as.data(), bs.data(), nullptr, &batch) ==
             MUSCLE_HIP_OK,
         "batch_create");
  if (batch) {
    for (int mode : {0, 0, 1, 2}) {
      for (auto& d : pairs)
        expect(hipMemset(d.dc, 0x7f, (size_t)d.cs.c.span * esize(d.dt)) == hipSuccess, "poison C", mode);
      expect(muscle_hip_batch_run(h, batch, mode) == MUSCLE_HIP_OK, "batch_run", mode);
      expect(muscle_hip_synchronize(h) == MUSCLE_HIP_OK, "batch synchronize", mode);
      for (size_t i = 0; i < pairs.size(); ++i) expect(dev_error(pairs[i]) <= 1e-12, "batch pair", (int64_t)i);
    }
    muscle_hip_batch_info_t bi;
    expect(muscle_hip_batch_get_info(batch, &bi) == MUSCLE_HIP_OK && bi.pairs == (int64_t)pairs.size(), "batch info");
    for (int64_t i = 0; i < (int64_t)pairs.size(); ++i) {
      muscle_hip_batch_pair_info_t pi;
      expect(muscle_hip_batch_get_pair_info(batch, i, &pi) == MUSCLE_HIP_OK, "pair info", i);
    }
    muscle_hip_batch_pair_info_t pi;
    expect(muscle_hip_batch_get_pair_info(batch, (int64_t)pairs.size(), &pi) != MUSCLE_HIP_OK, "pair index range");
    expect(muscle_hip_batch_destroy(batch) == MUSCLE_HIP_OK, "batch_destroy");
  }
  for (auto& d : pairs) free_dev_case(d);
  expect(muscle_hip_destroy(h) == MUSCLE_HIP_OK, "destroy handle");
  std::printf("gpu: %d contractions, a batch of %zu pairs in 4 runs\n", n_single, pairs.size());

  // server: chains ((x y) z) of ComplexF64 matrices, a few jobs at once
  muscle_hip_server_t srv = nullptr;
  expect(muscle_hip_server_create(int64_t(256) << 20, 4, 0, &srv) == MUSCLE_HIP_OK, "server_create");
  if (!srv) return;
  struct Job {
    int64_t d0, d1, d2, d3;
    std::vector<cd> X, Y, Z, want;
    void *dx, *dy, *dz;
    int64_t id;
  };
  std::vector<Job> jobs(12);
  const int32_t lx[2] = {1, 2}, ly[2] = {2, 3}, lz[2] = {3, 4};
  for (auto& j : jobs) {
    std::uniform_int_distribution<int> ud(1, 24);
    j.d0 = ud(rng);
    j.d1 = ud(rng);
    j.d2 = ud(rng);
    j.d3 = ud(rng);
    std::normal_distribution<double> nd;
    auto fill = [&](std::vector<cd>& v, int64_t n) {
      v.resize((size_t)n);
      for (auto& x : v) x = cd(nd(rng), nd(rng));
    };
    fill(j.X, j.d0 * j.d1);
    fill(j.Y, j.d1 * j.d2);
    fill(j.Z, j.d2 * j.d3);
    // want = (X Y) Z, column-major
    std::vector<cd> XY((size_t)(j.d0 * j.d2), cd(0, 0));
    for (int64_t a = 0; a < j.d0; ++a)
      for (int64_t c = 0; c < j.d2; ++c)
        for (int64_t b = 0; b < j.d1; ++b) XY[(size_t)(a + j.d0 * c)] += j.X[(size_t)(a + j.d0 * b)] * j.Y[(size_t)(b + j.d1 * c)];
    j.want.assign((size_t)(j.d0 * j.d3), cd(0, 0));
    for (int64_t a = 0; a < j.d0; ++a)
      for (int64_t d = 0; d < j.d3; ++d)
        for (int64_t c = 0; c < j.d2; ++c) j.want[(size_t)(a + j.d0 * d)] += XY[(size_t)(a + j.d0 * c)] * j.Z[(size_t)(c + j.d2 * d)];
    auto up = [&](const std::vector<cd>& v, void** dst) {
      const auto hb = encode(v, MUSCLE_HIP_C64);
      expect(hipMalloc(dst, hb.size()) == hipSuccess, "server leaf alloc");
      expect(hipMemcpy(*dst, hb.data(), hb.size(), hipMemcpyHostToDevice) == hipSuccess, "server leaf copy");
    };
    up(j.X, &j.dx);
    up(j.Y, &j.dy);
    up(j.Z, &j.dz);
    const int64_t ext[5] = {1, j.d0, j.d1, j.d2, j.d3};
    const int64_t sx[2] = {1, j.d0}, sy[2] = {1, j.d1}, sz[2] = {1, j.d2};
    const int64_t ex[2] = {j.d0, j.d1}, ey[2] = {j.d1, j.d2}, ez[2] = {j.d2, j.d3};
    muscle_hip_tensor_t leaves[3] = {{MUSCLE_HIP_C64, 2, j.dx, lx, ex, sx},
                                     {MUSCLE_HIP_C64, 2, j.dy, ly, ey, sy},
                                     {MUSCLE_HIP_C64, 2, j.dz, lz, ez, sz}};
    const int32_t lhs[2] = {0, 3}, rhs[2] = {1, 2}, off[3] = {0, 2, 4}, nmodes[4] = {1, 3, 1, 4};
    muscle_hip_job_t job{3, 2, leaves, lhs, rhs, off, nmodes, 5, ext};
    expect(muscle_hip_server_submit(srv, &job, &j.id) == MUSCLE_HIP_OK, "server_submit");
  }
  int done = 0;
  for (auto& j : jobs) {
    muscle_hip_job_result_t r;
    expect(muscle_hip_server_wait(srv, j.id, 120.0, &r) == MUSCLE_HIP_OK, "server_wait", j.id);
    if (r.status != MUSCLE_HIP_OK || r.result_elems != j.d0 * j.d3) {
      expect(false, "server job status", j.id);
      continue;
    }
    std::vector<char> buf((size_t)r.result_elems * 16);
    expect(muscle_hip_server_copy_result(srv, j.id, buf.data()) == MUSCLE_HIP_OK, "copy_result", j.id);
    std::vector<cd> got((size_t)r.result_elems);
    for (size_t i = 0; i < got.size(); ++i) got[i] = decode(buf, MUSCLE_HIP_C64, i);
    expect(rel_err(got, j.want) <= 1e-12, "server job result", j.id);
    expect(muscle_hip_server_release(srv, j.id) == MUSCLE_HIP_OK, "release", j.id);
    ++done;
  }
  muscle_hip_server_stats_t stats;
  expect(muscle_hip_server_get_stats(srv, &stats) == MUSCLE_HIP_OK && stats.completed == (int64_t)jobs.size(),
         "server stats");
  expect(muscle_hip_server_destroy(srv) == MUSCLE_HIP_OK, "server_destroy");
  for (auto& j : jobs) {
    expect(hipFree(j.dx) == hipSuccess && hipFree(j.dy) == hipSuccess && hipFree(j.dz) == hipSuccess, "hipFree");
  }
  std::printf("server: %d jobs checked\n", done);
}

}  // namespace

int main(int argc, char** argv) {
  std::mt19937_64 rng(20261203);
  check_describe(rng);
  std::mt19937_64 rng_k(20261204);
  check_ktiles(rng_k);
  check_fp32_ktiles();
  check_bits(rng_k);
  std::mt19937_64 rng_o(20261205);
  check_bits_offsets(rng_o);
  check_bits_empty();
  check_bits_rules();
  if (argc > 1 && std::strcmp(argv[1], "--gpu") == 0) check_gpu(rng);
  std::printf("%s: %d failures\n", g_failures ? "FAILED" : "ok", g_failures);
  return g_failures ? 1 : 0;
}
