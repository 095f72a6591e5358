// LDS-direct staging and MFMA operand reads of row-major bf16 / fp32 matrices
// for the Linears' products (esa_linear_gemm.hip, esa_wgrad.hip): a stage is
// 32 (bf16) or 16 (fp32) values of the contraction, 8 KB per 128 rows or
// columns of an operand, loaded 1 KB (64 lanes x 16 bytes) at a time.
#pragma once
#include "esa_attn_tiles.h"

namespace {

constexpr uint32_t kPastRange = 0xfffffff0u;   // a buffer offset past every range: loads give zeros, stores are dropped

DEVI f32x16 mfma32x2(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// The 18 wait states that v_mfma_f32_32x32x2_f32 (16 passes) asks for before a vector instruction touches its result,
// written out where that instruction stands in a block of its own that several paths reach: the compiler then counts
// the longest of them and has put none (a sum took an accumulator register before the matrix pipe had written it).
DEVI void mfma_settled(f32x16& acc) { asm volatile("s_nop 15\n\ts_nop 1" : "+v"(acc)); }

// An operand whose contraction runs over the rows in memory, staged as [rows
// of the stage][COLS]: the operands of dW = g^T x (rows = tokens) and W in
// dx = g W.  bf16 operands come from ds_read_b64_tr_b16, and a row's 16-byte
// chunk c sits in slot c ^ 2 (row mod 4), which spreads the four rows of a
// transpose read over the banks.
template <typename T, int COLS>
struct Rows;
template <int COLS>
struct Rows<bf16, COLS> {
  static constexpr int kTok = 32, kSteps = 2;   // tokens per stage, MFMA k steps of it
  static constexpr int kBytes = kTok * COLS * 2, kLoads = kBytes / 4096;   // 1 KB LDS-direct loads per wave
  typedef bf16x8 Op;
  // lane's byte offset (in the stage's 1 KB load j) from the stage's first row
  static DEVI uint32_t offset(int j, int lane, int col0, int cols) {
    constexpr int kChunks = COLS / 8;   // 16-byte chunks per row
    const int tok = (64 * j + lane) / kChunks, slot = (64 * j + lane) % kChunks, c = col0 + 8 * (slot ^ (2 * (tok & 3)));
    return c < cols ? (uint32_t)(tok * cols + c) * 2u : kPastRange;
  }
  // features c0 .. c0 + 31 over the 16 tokens of step k
  static DEVI Op operand(const char* lds, int c0, int k, int lane) {
    const int i = lane & 15, grp = lane >> 4;
    const int tok = 16 * k + 8 * (grp >> 1) + (i >> 2), c = c0 + 16 * (grp & 1) + 4 * (i & 3);
    const int slot = (c >> 3) ^ (2 * (tok & 3));
    const bf16* p = reinterpret_cast<const bf16*>(lds) + tok * COLS + slot * 8 + (c & 4);
    const bf16x4 lo = lds_tr4(p), hi = lds_tr4(p + 4 * COLS);   // tokens + 4: the same slot
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
  static DEVI f32x16 product(const Op& a, const Op& b, const f32x16& c) { return mfma32(a, b, c); }
  static DEVI float add_tokens(const Op& a, float s) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 one = {(bf16)1.f, (bf16)1.f};
#pragma unroll
    for (int e = 0; e < 8; e += 2) s = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{a[e], a[e + 1]}, one, s, false);
    return s;
  }
};
template <int COLS>
struct Rows<float, COLS> {
  static constexpr int kTok = 16, kSteps = 8;
  static constexpr int kBytes = kTok * COLS * 4, kLoads = kBytes / 4096;
  typedef float Op;
  static DEVI uint32_t offset(int j, int lane, int col0, int cols) {
    constexpr int kChunks = COLS / 4;
    const int tok = (64 * j + lane) / kChunks, c = col0 + 4 * ((64 * j + lane) % kChunks);
    return c < cols ? (uint32_t)(tok * cols + c) * 4u : kPastRange;
  }
  static DEVI Op operand(const char* lds, int c0, int k, int lane) {
    return reinterpret_cast<const float*>(lds)[(2 * k + (lane >> 5)) * COLS + c0 + (lane & 31)];
  }
  static DEVI f32x16 product(const Op& a, const Op& b, const f32x16& c) { return mfma32x2(a, b, c); }
  static DEVI float add_tokens(const Op& a, float s) { return s + a; }
};

// An operand whose contraction runs along the rows in memory, staged as
// [LINES rows][64 bytes]: x and W in y = x W^T, g in dx = g W.  Two rows share
// a 128-byte line; chunk c of a row sits in slot c ^ (line mod 4) of its half,
// so eight lanes reading one chunk of consecutive rows touch eight 16-byte slots.
template <int LINES>
struct Along {
  static constexpr int kBytes = LINES * 64, kLoads = kBytes / 4096;   // 1 KB loads per wave
  // lane's byte offset (in the stage's 1 KB load j) from the stage's first row, rows `pitch` bytes apart
  static DEVI uint32_t offset(int j, int lane, int pitch) {
    const int p = 64 * j + lane, line = p >> 3, row = 2 * line + ((p >> 2) & 1);
    return (uint32_t)(row * pitch + 16 * ((p & 3) ^ (line & 3)));
  }
  static DEVI const char* chunk(const char* lds, int row, int c) {
    return lds + (row >> 1) * 128 + (row & 1) * 64 + ((c ^ ((row >> 1) & 3)) << 4);
  }
};

}  // namespace
