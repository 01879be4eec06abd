// Contractions whose extents are all powers of two and that do little work
// per output (K short, or an output side short): tiles of C in address order.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "lowering.hpp"

namespace mh {

// Sizes of the kernel: 256 threads, 8 outputs each (a tile of 2^11 outputs).
constexpr int kBitLane = 6, kBitThread = 8, kBitReg = 3, kBitTile = kBitThread + kBitReg;
constexpr int kBitLongIt = 8, kBitShortIt = 4;  // elements each thread gathers per K chunk at most
constexpr int kBitOuter = 32, kBitChunk = 12;

// One contraction.  With power-of-two extents every offset is the sum of what
// the index bits contribute, so a tile needs no offset table: the low bits of
// an output's number inside the tile are the thread's, the next three its
// registers', and a tile's number gives the rest.  The long operand is the one
// with more elements in a tile (LDS region 0), the short one the other.
// Element strides; LDS contributions combine by exclusive or.
struct BitDesc {
  const void* L;  // long operand
  const void* S;  // short operand
  void* C;
  int32_t reg_long;  // register bits that select the long operand's element (the others select the short one's)
  int32_t long_b;    // the long operand is the second one
  int32_t run;       // consecutive tiles per workgroup
  int32_t tiles;
  int32_t kc, nchunk;  // K elements per chunk, chunks
  int32_t c_stream;
  int32_t line_k;      // (host) bits of K inside a 128-byte line of the long operand,
  int32_t line_split;  // and whether some of them belong to another chunk
  int32_t nl, ns;                // elements of a K chunk in the long and short operands (powers of two)
  int32_t sl, ss;                // LDS elements per k of each
  int32_t kxl, kxs;              // k bits folded into the low LDS bits of each
  uint32_t tC[kBitThread], tL[kBitThread], tS[kBitThread];  // thread bits: C stride, LDS of the operands
  uint32_t rC[kBitReg], rX[kBitReg];                        // register bits (the long operand's first): C stride, LDS
  // gathers, in the operand's own address order: thread bits, then iterations
  uint32_t gL[kBitThread], gLl[kBitThread], gS[kBitThread], gSl[kBitThread];
  uint32_t iL[kBitLongIt], iLl[kBitLongIt], iS[kBitShortIt], iSl[kBitShortIt];
  uint32_t oL[kBitOuter], oS[kBitOuter], oC[kBitOuter];  // tile number bits
  // steps from a tile (K chunk) number whose low j bits are ones to the next
  uint32_t sL[4], sS[4], sC[4];
  uint32_t cL[kBitChunk], cS[kBitChunk];
};

struct BitArgs {
  const BitDesc* descs;
  const int2* items;  // (contraction, first tile)
  int64_t nitems;
};

// Plans a lowered contraction for the kernel above; false when it does not
// apply (another kernel then takes it).  Operand addresses are left out.
bool plan_bits(const ContractionDesc& d, BitDesc& out);

// One contraction (the plain call), or the items of a batch
void launch_bits_one(bool dbl, bool cplx, const BitDesc& d, hipStream_t s);
// (lds_elems: the largest nl + ns among them).
void launch_bits(bool dbl, bool cplx, const BitArgs& a, int lds_elems, hipStream_t s);

}  // namespace mh
