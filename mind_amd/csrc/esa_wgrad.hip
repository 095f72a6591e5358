// Weight and bias gradients of the packed blocks' Linear layers on gfx950:
// dW_i = g_i^T x_i and db_i = column sums of g_i, for up to eight (g_i, x_i)
// over the same rows (a block's nn.Linears, esa/mha.py:12-15, 54-56,
// esa/mlp_utils.py:18-37, in one launch or one by one), g_i [rows, out]
// and x_i [rows, in] both bf16 or both fp32, results fp32.
//
// The contraction runs over the tokens (up to hundreds of thousands) into a
// small matrix, so it is cut over the rows: block = one 128 x 128 (bf16 also
// 128 x 256) tile of one dW over one range of rows, the partial tiles added by
// a second launch in a fixed order (deterministic, no atomics).  What bounds it
// is reading g and x once from HBM where the matrix is one tile, and the LDS
// reads of the operands beside the MFMAs where it is many.
//
// Both operands need the token dimension in the MFMA K slots while the rows
// in memory run over features.  bf16: v_mfma_f32_32x32x16_bf16, operands by
// ds_read_b64_tr_b16 (four tokens of 16 features per read) from rows staged
// as they are in memory; fp32: v_mfma_f32_32x32x2_f32, whose operand is one
// value per lane, so a plain 4-byte read of 32 consecutive features serves.
// Rows are staged 32 (bf16) or 16 (fp32) tokens at a time by LDS-direct
// loads, three stage buffers deep, one barrier per stage; rows and columns
// past the end lie past the buffer range and load zeros.  A bf16 row's
// 16-byte chunk c sits in slot c ^ 2 (token mod 4), which spreads the four
// tokens of a transpose read over the banks.  Four waves of 64 x 64, or of 64 x
// 128 where the block's tile is 128 x 256 (64 or 128 accumulator registers).
// The bias sums ride on the operand registers the tile's first column block
// holds anyway (v_dot2_f32_bf16 against ones).
//
// Measured against the token-chunk GEMMs of the library with their sum, the
// leftover rows' GEMM and the column sum kernels (weight and bias gradient,
// us): bf16 33,000 x 256 x 256 20 vs 49, three of them 29 vs 147; 43,670 x
// 768 x 192 29 vs 94; 129,850 x 512 x 512 94 vs 139 (724 TFLOP/s); 129,850 x
// 2048 x 512 284 vs 381 (958 TFLOP/s); fp32 21,752 x 128 x 128 23 vs 54,
// three 34 vs 162; 33,000 x 1024 x 256 141 vs 160 (123 of the 154 TFLOP/s that
// a large fp32 product reaches).  The six weights of a SAB block with its MLP
// in one launch: fp32 21,752 x 128 63 vs 105 in four, bf16 33,000 x 256 56 vs 99.  The stage loop holds no spill and no copy of
// the accumulators: scratch loads share the counter that the staging waits on,
// and a spilling first version ran at a third of the rate.
#include <algorithm>
#include <type_traits>

#include "esa_stage.h"
#include "esa_profile.h"
#include "../../include/esa_hip.h"

namespace {

constexpr int kMaxPairs = 8;
constexpr int kWTileO = 128;                 // block tile along `out` (two waves of 64); along `in`: 64 NV (two of 32 NV)
constexpr int kStages = 3;
constexpr int kCus = 256, kMinRows = 128;
// The bias sums of this many stages are added to those before them, instead of a row range's tokens in one chain
// (relative error against 64 bits, fp32 21,752 x 128: 2.05e-7 in one chain, 1.44 here, 1.76 in the column sum;
// 129,850 x 512: 7.7, 1.9 and 2.5e-7).
constexpr int kBiasFold = 4;
// In fp32 ranges of more than kFoldRows rows the sums of kFold stages are added to those before them, too (FOLD):
// 129,850 x 2048 x 512, 16,256 rows a range: 2.3e-6 in one chain, 4.2e-7 folded, the library's token-chunk products
// 1.6e-6.  It takes 50 registers and 4 % (2,005 -> 2,086 us; shorter ranges by more splits: 2,450), which ranges up to
// 4,096 rows are spared: 1.1e-6 in one chain.
constexpr int kFold = 32, kFoldRows = 4096;

struct WgradPair {
  const void* g; const void* x;
  float* part;    // [splits][out][in]
  float* bpart;   // [splits][out], or null
  int out, in, tiles_i, tile0;   // tile0: first tile of this pair among all pairs' tiles
};
struct WgradArgs {
  int rows, chunk, tiles, n;
  WgradPair p[kMaxPairs];
};

struct ReducePart { const float* src; float* dst; int64_t n; int block0; };
struct ReduceArgs { int splits, n; ReducePart p[2 * kMaxPairs]; };

template <typename T, int NV, bool FOLD>
__global__ __launch_bounds__(256, 2) void wgrad_kernel(const WgradArgs a) {
  constexpr int kTileI = 64 * NV;
  using RG = Rows<T, kWTileO>;
  using RX = Rows<T, kTileI>;
  constexpr int kTok = RG::kTok, kSteps = RG::kSteps;
  __shared__ __align__(16) char lds[kStages][RG::kBytes + RX::kBytes];
  // XCD-contiguous order, tiles of one row range side by side: they read the same rows
  const int G = (int)gridDim.x, hb = (int)blockIdx.x, xcd = hb & 7, q = G >> 3, rem = G & 7;
  const int item = xcd * q + min(xcd, rem) + (hb >> 3);
  const int split = item / a.tiles, tile = item - split * a.tiles;
  int pi = 0;
#pragma unroll
  for (int i = 1; i < kMaxPairs; ++i)
    if (i < a.n && tile >= a.p[i].tile0) pi = i;
  const WgradPair p = a.p[pi];
  const int to = (tile - p.tile0) / p.tiles_i, ti = (tile - p.tile0) - to * p.tiles_i;
  const int o0 = to * kWTileO, i0 = ti * kTileI;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wo = 64 * (wave >> 1), wi = 32 * NV * (wave & 1);
  const int t0 = split * a.chunk, nt = min(a.chunk, a.rows - t0);   // nt > 0
  const T* g = (const T*)p.g + (size_t)t0 * p.out;
  const T* x = (const T*)p.x + (size_t)t0 * p.in;
  const int stages = (nt + kTok - 1) / kTok;
  uint32_t goff[RG::kLoads], xoff[RX::kLoads];   // this lane's chunk in the wave's loads of a stage
#pragma unroll
  for (int j = 0; j < RG::kLoads; ++j) goff[j] = RG::offset(RG::kLoads * wave + j, lane, o0, p.out);
#pragma unroll
  for (int j = 0; j < RX::kLoads; ++j) xoff[j] = RX::offset(RX::kLoads * wave + j, lane, i0, p.in);
  auto load = [&](int s, int buf) {   // the range's rows from stage s on as the buffer: rows past it load zeros
    const int t = s * kTok;
    const rsrc_t rg = make_rsrc(g + (size_t)t * p.out, (uint32_t)(nt - t) * p.out * sizeof(T));
    const rsrc_t rx = make_rsrc(x + (size_t)t * p.in, (uint32_t)(nt - t) * p.in * sizeof(T));
#pragma unroll
    for (int j = 0; j < RG::kLoads; ++j) dma16(rg, goff[j], lds[buf] + 1024 * (RG::kLoads * wave + j));
#pragma unroll
    for (int j = 0; j < RX::kLoads; ++j) dma16(rx, xoff[j], lds[buf] + RG::kBytes + 1024 * (RX::kLoads * wave + j));
  };
  const bool live = o0 + wo < p.out && i0 + wi < p.in;   // wave-uniform: a wave wholly past the matrix only loads
  const bool bias = p.bpart && ti == 0 && wi == 0;
  f32x16 acc[2][NV];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[u][v] = f32x16{};
  float bs[2] = {0.f, 0.f}, bias_sum[2] = {0.f, 0.f};   // of the last stages, of those before them
  f32x16 sum[FOLD ? 2 : 1][FOLD ? NV : 1] = {};         // of acc and bias_sum, before the last kFold stages
  float bias_before[2] = {0.f, 0.f};
  // One stage's products; all operands of the stage are read first, so the reads of a step overlap the last one's MFMAs.
  auto multiply = [&](int buf, int stage, auto with_bias) {
    typename RG::Op og[kSteps][2], ox[kSteps][NV];
#pragma unroll
    for (int k = 0; k < kSteps; ++k) {
#pragma unroll
      for (int u = 0; u < 2; ++u) og[k][u] = RG::operand(lds[buf], wo + 32 * u, k, lane);
#pragma unroll
      for (int v = 0; v < NV; ++v) ox[k][v] = RX::operand(lds[buf] + RG::kBytes, wi + 32 * v, k, lane);
    }
#pragma unroll
    for (int k = 0; k < kSteps; ++k) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[u][v] = RG::product(og[k][u], ox[k][v], acc[u][v]);
      if constexpr (with_bias.value)
#pragma unroll
        for (int u = 0; u < 2; ++u) bs[u] = RG::add_tokens(og[k][u], bs[u]);
    }
    if (with_bias.value && stage % kBiasFold == kBiasFold - 1)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bias_sum[u] += bs[u];
        bs[u] = 0.f;
      }
    if constexpr (FOLD)
      if (stage % kFold == kFold - 1)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          bias_before[u] += bias_sum[u];
          bias_sum[u] = 0.f;
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            mfma_settled(acc[u][v]);
#pragma unroll
            for (int e = 0; e < 16; ++e) sum[u][v][e] += acc[u][v][e];
            acc[u][v] = f32x16{};
          }
        }
  };
  // Every wave runs the same stages and barriers; `use` is what it does with a stage.
  auto run = [&](auto use) {
    load(0, 0);
    if (stages > 1) load(1, 1);
    for (int s0 = 0; s0 < stages; s0 += kStages) {
#pragma unroll
      for (int buf = 0; buf < kStages; ++buf) {
        const int s = s0 + buf;
        if (s >= stages) break;
        if (s + 1 < stages) wait_vmcnt<RG::kLoads + RX::kLoads>();   // this wave's loads of stage s have landed
        else wait_vmcnt<0>();
        __syncthreads();   // every wave's have, and every wave is done with stage s - 1, whose buffer is loaded next
        if (s + 2 < stages) load(s + 2, (buf + 2) % kStages);
        use(buf, s);
      }
    }
  };
  if (!live) run([](int, int) {});
  else if (bias) run([&](int buf, int s) { multiply(buf, s, std::true_type{}); });
  else run([&](int buf, int s) { multiply(buf, s, std::false_type{}); });
  if (!live) return;
  if constexpr (FOLD)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        mfma_settled(acc[u][v]);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[u][v][e] += sum[u][v][e];
      }
  const int col = lane & 31, half = lane >> 5;
  // rows past `out` lie past the buffer, columns past `in` are sent there: both stores are dropped
  const rsrc_t ro = make_rsrc(p.part + (size_t)split * p.out * p.in, (uint32_t)p.out * p.in * 4u);
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = i0 + wi + 32 * v + col;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = o0 + wo + 32 * u + 8 * (r >> 2) + 4 * half + (r & 3);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[u][v][r]), ro,
                                              i < p.in ? (uint32_t)(o * p.in + i) * 4u : 0xfffffff0u, 0, 0);
      }
    }
  if (bias)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float b = bias_before[u] + (bias_sum[u] + bs[u]);
      const float sum_b = b + __shfl_xor(b, 32);   // the lane halves hold different tokens
      const int o = o0 + wo + 32 * u + col;
      if (half == 0 && o < p.out) p.bpart[(size_t)split * p.out + o] = sum_b;
    }
}

// dst[e] = sum over the splits of src[split][e]: in split order within eights
// of four interleaved slices, the eights in order, then the slices (bf16
// 500,000 x 64: the bias sum 2.0e-7 from 64 bits with a slice in one chain,
// 1.0e-7 so, 1.5e-7 as a column sum).  A block takes 256 values,
// four per lane, one slice per wave: the loads of a wave's slice are
// independent of its adds, and small matrices still fill the chip.
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const ReduceArgs a) {
  __shared__ __align__(16) f32x4 sums[3][64];
  int pi = 0;
#pragma unroll
  for (int i = 1; i < 2 * kMaxPairs; ++i)
    if (i < a.n && (int)blockIdx.x >= a.p[i].block0) pi = i;
  const ReducePart p = a.p[pi];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t e = ((int64_t)((int)blockIdx.x - p.block0) * 64 + lane) * 4;
  f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
  if (e < p.n) {
    for (int k0 = wave; k0 < a.splits; k0 += 32) {   // eight at a time, their loads in flight together
      f32x4 v[8], part = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = *reinterpret_cast<const f32x4*>(p.src + (size_t)min(k0 + 4 * i, a.splits - 1) * p.n + e);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) part[j] += k0 + 4 * i < a.splits ? v[i][j] : 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += part[j];
    }
  }
  if (wave) sums[wave - 1][lane] = s;
  __syncthreads();
  if (wave == 0 && e < p.n) {
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const f32x4 v = sums[w][lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += v[j];
    }
    *reinterpret_cast<f32x4*>(p.dst + e) = s;
  }
}

struct WgradSplit { int splits, chunk, tiles, nv; };

// Row ranges and the tile width.  Ranges: two blocks per CU, one below that
// (a CU with two blocks beside CUs with one would be the launch's end: fp32
// 21,752 x 256 x 128, 340 -> 256 blocks, 31.5 -> 24.8 us), none shorter than
// kMinRows rows, whose staging would not be in flight long enough to pay for
// its partial tile (64 rows: bf16 33,000 x 256 x 256 19.9 -> 27.0 us); a
// range's rows stay within 1 GiB of buffer offsets.  Width: 256 columns for
// bf16 where three weights of 512 x 512 or more leave a wide tile long ranges
// (its LDS reads per product are a quarter fewer, its partials twice as large:
// 129,850 x 2048 x 512 318 -> 284 us, three of 512 x 512 289 -> 236 us, but
// 33,000 x 1024 x 256 32 -> 41 us).
WgradSplit wgrad_split(int64_t rows, int n, const int* out, const int* in, int elem) {
  auto tiles = [&](int nv) {
    int t = 0;
    for (int i = 0; i < n; ++i) t += ((out[i] + kWTileO - 1) / kWTileO) * ((in[i] + 64 * nv - 1) / (64 * nv));
    return t;
  };
  WgradSplit w{1, 1, tiles(2), 2};
  if (elem == 2 && tiles(4) >= 24 && rows >= 16384) w.nv = 4, w.tiles = tiles(4);
  int64_t widest = 1;
  for (int i = 0; i < n; ++i) widest = std::max<int64_t>(widest, std::max(out[i], in[i]));
  const int64_t most = std::max<int64_t>(1, rows / kMinRows);
  const int blocks = most * w.tiles >= 2 * kCus ? 2 * kCus : kCus;
  const int64_t s = std::max<int64_t>({1, std::min<int64_t>(blocks / w.tiles, most), (rows * widest * elem >> 30) + 1});
  w.chunk = (int)std::max<int64_t>(32, ((rows + s - 1) / s + 31) / 32 * 32);
  w.splits = (int)std::max<int64_t>(1, (rows + w.chunk - 1) / w.chunk);
  return w;
}

bool wgrad_misaligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; }

int wgrad_check(int64_t rows, int n, const int* out, const int* in, int dtype) {
  if (n < 1 || n > kMaxPairs || rows < 0 || rows > 0x7fffffff) return ESA_ERR_SHAPE;
  if (dtype != ESA_F32 && dtype != ESA_BF16) return ESA_ERR_DTYPE;
  if (!out || !in) return ESA_ERR_NULL;
  const int unit = dtype == ESA_BF16 ? 8 : 4;   // 16-byte row chunks
  for (int i = 0; i < n; ++i)
    if (out[i] < unit || in[i] < unit || out[i] % unit || in[i] % unit || out[i] > 16384 || in[i] > 16384)
      return ESA_ERR_SHAPE;
  return ESA_OK;
}

size_t wgrad_bytes(const WgradSplit& w, int n, const int* out, const int* in) {
  size_t b = 0;
  if (w.splits > 1)
    for (int i = 0; i < n; ++i) b += (size_t)w.splits * ((size_t)out[i] * in[i] + out[i]) * sizeof(float);
  return b;
}

}  // namespace

extern "C" {

int esa_weight_grad_workspace_size(long long rows, int n, const int* out_features, const int* in_features, int dtype,
                                   size_t* bytes) {
  if (!bytes) return ESA_ERR_NULL;
  if (const int rc = wgrad_check(rows, n, out_features, in_features, dtype)) return rc;
  *bytes = wgrad_bytes(wgrad_split(rows, n, out_features, in_features, dtype == ESA_BF16 ? 2 : 4), n, out_features,
                       in_features);
  return ESA_OK;
}

int esa_weight_grad(long long rows, int n, const void* const* g, const void* const* x, const int* out_features,
                    const int* in_features, int dtype, float* const* dw, float* const* db, void* workspace,
                    size_t workspace_bytes, void* stream) {
  if (const int rc = wgrad_check(rows, n, out_features, in_features, dtype)) return rc;
  if (!g || !x || !dw || !db) return ESA_ERR_NULL;
  if (rows < 1) return ESA_ERR_SHAPE;
  const WgradSplit w = wgrad_split(rows, n, out_features, in_features, dtype == ESA_BF16 ? 2 : 4);
  if (workspace_bytes < wgrad_bytes(w, n, out_features, in_features)) return ESA_ERR_WORKSPACE;
  if (w.splits > 1 && !workspace) return ESA_ERR_NULL;
  if (w.splits > 1 && wgrad_misaligned(workspace)) return ESA_ERR_ALIGN;
  WgradArgs a{};
  ReduceArgs r{};
  a.rows = (int)rows; a.chunk = w.chunk; a.tiles = w.tiles; a.n = n;
  r.splits = w.splits;
  float* ws = (float*)workspace;
  int tile = 0;
  int64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    const int o = out_features[i], in = in_features[i], ti = (in + 64 * w.nv - 1) / (64 * w.nv);
    if (!g[i] || !x[i] || !dw[i]) return ESA_ERR_NULL;
    if (wgrad_misaligned(g[i]) || wgrad_misaligned(x[i]) || wgrad_misaligned(dw[i]) || wgrad_misaligned(db[i]))
      return ESA_ERR_ALIGN;
    WgradPair p{g[i], x[i], dw[i], db[i], o, in, ti, tile};
    tile += ti * ((o + kWTileO - 1) / kWTileO);
    if (w.splits > 1) {
      p.part = ws;
      ws += (size_t)w.splits * o * in;
      r.p[r.n++] = ReducePart{p.part, dw[i], (int64_t)o * in, (int)blocks};
      blocks += ((int64_t)o * in + 255) / 256;
      if (db[i]) {
        p.bpart = ws;
        ws += (size_t)w.splits * o;
        r.p[r.n++] = ReducePart{p.bpart, db[i], o, (int)blocks};
        blocks += (o + 255) / 256;
      }
    }
    a.p[i] = p;
  }
  const int64_t items = (int64_t)w.tiles * w.splits;
  if (items > 0x7fffffffLL || blocks > 0x7fffffffLL) return ESA_ERR_SHAPE;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define ESA_WGRAD(T, NV, FOLD) \
  ESA_TIMED(esa_profile::kWeightGrad, st, \
            hipLaunchKernelGGL((wgrad_kernel<T, NV, FOLD>), dim3((unsigned)items), dim3(256), 0, st, a))
  if (dtype == ESA_F32 && w.chunk > kFoldRows) ESA_WGRAD(float, 2, true);
  else if (dtype == ESA_F32) ESA_WGRAD(float, 2, false);
  else if (w.nv == 4) ESA_WGRAD(bf16, 4, false);
  else ESA_WGRAD(bf16, 2, false);
#undef ESA_WGRAD
  ESA_LAUNCH_CHECK();
  if (w.splits > 1) {
    ESA_TIMED(esa_profile::kWeightGrad, st,
              hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, st, r));
    ESA_LAUNCH_CHECK();
  }
  return ESA_OK;
}

}  // extern "C"
