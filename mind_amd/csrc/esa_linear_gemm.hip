// The blocks' Linears with what follows them, and their input gradients, on
// gfx950 (esa_linear_fwd, esa_linear_dx; bf16 or fp32):
//   y_i = x W_i^T + b_i for up to three weights over one input, or for one:
//   z and mish(z) (an MLP's Linear -> Mish, esa/mlp_utils.py:18-37),
//   z and o + mish(z), plus the block's residual (esa/mha.py:87,
//   esa/masked_layers.py:471-472), or r(y) + residual (:478-483);
//   dx = [base +] sum_i g_i W_i over up to three pairs (fc_q / fc_k / fc_v
//   share their input, esa/mha.py:54-56), or (g W) mish'(z).
// A library GEMM reaches the large shapes' rate, but its call costs about 18
// us of host time (10-40 us are the kernels of a small batch) and the element-
// wise passes around it read and write what its epilogue holds in registers.
//
// Block = 64 TT tokens x 64 NV features, four waves of 32 TT x 32 NV: 64 x 64
// in fp32 and on small bf16 launches, else 128 x 128 or 256 (gemm_tile).
// Operands are staged by LDS-direct loads (esa_stage.h), 64 bytes of the
// contraction per row and stage, three buffers deep, one barrier per stage.  bf16:
// v_mfma_f32_32x32x16_bf16 with the features as the MFMA's rows, so that a
// lane holds four consecutive features of a token; the 32-token halves of the
// accumulators pass through the wave's part of the (then free) stage buffers
// in fp32 and leave as 16-byte rows, the epilogue's other inputs read the same
// way.  fp32: v_mfma_f32_32x32x2_f32, the same otherwise.
//
// What bounds it: latency of a few stages on small batches, the epilogue's
// memory passes at widths near the contraction, the LDS reads beside the MFMAs
// (about 900 TFLOP/s) at large ones.  Against the library GEMM and the passes
// it replaces (us, back to back): bf16 1,806 rows, 128 -> 128, 9 vs 21, with
// Mish 10.6 vs 27, three outputs 12.5 vs 61; 33,000 rows, 256 -> 256, with the
// MAB's residual 23.5 vs 30, with the block's 19 vs 78; 129,850 rows, 512 ->
// 512: 230 vs 235 and 195 vs 240, dx of three 196 vs 284, dx times the slope of
// a hidden layer of 2048 530 vs 628; fp32 21,752 rows, 128 -> 128, 12.5 vs 21,
// three outputs 28 vs 42.  Plain products of 4e10 operations and more run
// faster in the library (129,850 rows, 512 -> 2048: 320 vs 410), and the
// callers leave those to it.
#include <algorithm>

#include "esa_mish.h"
#include "esa_profile.h"
#include "esa_stage.h"
#include "../../include/esa_hip.h"

namespace {

constexpr int kGemmMax = 3, kGemmStages = 3;
// fp32 sums 128 values of a term (eight stages) from zero and adds that to the sums before it, as a product of that
// length or the library's term by term rounds, and not along the whole contraction.  Relative error against 64 bits of
// dx of three, 384 long: 3.0e-7 in one chain, 2.05e-7 here and in the library; 1,536 long 6.0, 2.1 and 4.0e-7;
// y 2,048 long 5.9, 1.6 and 5.9e-7.  It costs 0-4 % (21,752 rows, 128 -> 128: 12.6 -> 12.6 us, dx of three 26.0 -> 27.1);
// every 64 values took 2-6 %.
constexpr int kFold = 8;

// What follows the product; kDx*: the input gradient.
enum Epi { kPlain, kMish, kMab, kMabResidual, kAdd, kDx, kDxBase, kDxMish };
constexpr bool is_dx(int epi) { return epi >= kDx; }

struct GemmPart {   // an output of the forward, a term of dx
  const void* a;    // dx: g [rows, k]
  const void* w;    // [k' , in]: the Linear's weight
  const void* bias; // forward, or null
  void* y;          // forward: [rows, cols], null: not stored
  int k;            // contraction length
  int cols;         // forward: out_features
  int tile0;        // forward: first column tile
};
struct GemmArgs {
  int rows, n, col_tiles;
  int cols;             // dx: in_features
  const void* x;        // forward: [rows, k]
  const void* other;    // kMab*: o; kDxBase: base; kDxMish: z
  const float* residual;
  void* result;         // the epilogue's result, dx
  GemmPart p[kGemmMax];
};

template <typename T> struct Elem;
template <> struct Elem<bf16> { static constexpr int kStage = 32; };
template <> struct Elem<float> { static constexpr int kStage = 16; };

DEVI f32x4 load4f(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
DEVI f32x4 load4f(const bf16* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
// Eight values of a row (fp32 rows may end after four).
DEVI void load8f(f32x4 (&v)[2], const float* p, bool wide) {
  v[0] = load4f(p);
  if (wide) v[1] = load4f(p + 4);
}
DEVI void load8f(f32x4 (&v)[2], const bf16* p, bool) {
  const bf16x8 x = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e >> 2][e & 3] = (float)x[e];
}
DEVI void store8f(float* p, const f32x4 (&v)[2], bool wide) {
  *reinterpret_cast<f32x4*>(p) = v[0];
  if (wide) *reinterpret_cast<f32x4*>(p + 4) = v[1];
}
DEVI void store8f(bf16* p, const f32x4 (&v)[2], bool) {
  bf16x8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (bf16)v[e >> 2][e & 3];
  *reinterpret_cast<bf16x8*>(p) = x;
}

// One value of the result from the product (bias and base included) and the epilogue's inputs; z: the stored
// pre-activation, which the kernels that read it back see rounded.
template <typename T, int EPI>
DEVI float finish(float v, float other, float residual, float& z) {
  if constexpr (EPI == kMish || EPI == kMab || EPI == kMabResidual) {
    z = (float)(T)v;
    const float m = mish_f(z);
    if constexpr (EPI == kMish) return m;
    if constexpr (EPI == kMab) return other + m;
    return residual + (float)(T)(other + m);
  } else if constexpr (EPI == kAdd) {
    return (float)(T)v + residual;
  } else if constexpr (EPI == kDxMish) {
    return (float)(T)v * mish_grad_f(other);
  } else {
    return v;
  }
}

template <typename T, int TT, int NV, int EPI>
__global__ __launch_bounds__(256, 2) void linear_gemm_kernel(const GemmArgs a) {
  constexpr bool DX = is_dx(EPI), F32 = sizeof(T) == 4;
  constexpr int kTokTile = 64 * TT, kFeat = 64 * NV, KS = Elem<T>::kStage;
  using RA = Along<kTokTile>;
  using RW = Along<kFeat>;
  using RT = Rows<T, kFeat>;
  constexpr int kWBytes = DX ? RT::kBytes : RW::kBytes, kWLoads = DX ? RT::kLoads : RW::kLoads;
  constexpr int kWaveOut = 32 * 32 * NV * 4;   // the fp32 tile of 32 tokens that a wave's results pass through
  constexpr int kBuf = RA::kBytes + kWBytes;
  static_assert(4 * kWaveOut <= kGemmStages * kBuf, "epilogue tiles fit the stage buffers");
  __shared__ __align__(16) char lds[kGemmStages * kBuf];
  // XCD-contiguous order, the column tiles of one token block side by side: they read the same rows
  const int G = (int)gridDim.x, hb = (int)blockIdx.x, xcd = hb & 7, qq = G >> 3, rem = G & 7;
  const int item = xcd * qq + min(xcd, rem) + (hb >> 3);
  const int rb = item / a.col_tiles, ct = item - rb * a.col_tiles;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int row0 = rb * kTokTile, nrows = min(kTokTile, a.rows - row0);
  int part = 0;
  if constexpr (!DX) {
#pragma unroll
    for (int i = 1; i < kGemmMax; ++i)
      if (i < a.n && ct >= a.p[i].tile0) part = i;
  }
  const int f0 = (DX ? ct : ct - a.p[part].tile0) * kFeat, cols = DX ? a.cols : a.p[part].cols;
  const int wt = 32 * TT * (wave >> 1), wf = 32 * NV * (wave & 1);
  const bool live = wt < nrows && f0 + wf < cols;   // wave-uniform: a wave wholly past the result only loads

  int stages = 0;
  if constexpr (DX) {
    for (int i = 0; i < a.n; ++i) stages += a.p[i].k / KS;
  } else {
    stages = a.p[0].k / KS;
  }
  // The staged tensors' position: stage s0.. of a term (dx walks its terms one after another).
  int term = DX ? 0 : part, k0 = 0;
  uint32_t woff[kWLoads];
#pragma unroll
  for (int j = 0; j < kWLoads; ++j)
    woff[j] = DX ? RT::offset(kWLoads * wave + j, lane, f0, cols)
                 : RW::offset(kWLoads * wave + j, lane, a.p[part].k * (int)sizeof(T));
  auto load = [&](int buf) {
    const GemmPart& p = a.p[term];
    const int K = p.k;
    char* b = lds + buf * kBuf;
    const T* rows = (const T*)(DX ? p.a : a.x) + (size_t)row0 * K + k0;
    const rsrc_t ra = make_rsrc(rows, (uint32_t)(nrows * K - k0) * sizeof(T));
#pragma unroll
    for (int j = 0; j < RA::kLoads; ++j)
      dma16(ra, RA::offset(RA::kLoads * wave + j, lane, K * (int)sizeof(T)), b + 1024 * (RA::kLoads * wave + j));
    if constexpr (DX) {   // W [K, cols]: rows k0 .. of it
      const rsrc_t rw = make_rsrc((const T*)p.w + (size_t)k0 * cols, (uint32_t)(K - k0) * cols * sizeof(T));
#pragma unroll
      for (int j = 0; j < kWLoads; ++j) dma16(rw, woff[j], b + RA::kBytes + 1024 * (kWLoads * wave + j));
    } else {              // W [cols, K]: rows f0 .., columns k0 ..
      const rsrc_t rw = make_rsrc((const T*)p.w + (size_t)f0 * K + k0,
                                  (uint32_t)(min(kFeat, cols - f0) * K - k0) * sizeof(T));
#pragma unroll
      for (int j = 0; j < kWLoads; ++j) dma16(rw, woff[j], b + RA::kBytes + 1024 * (kWLoads * wave + j));
    }
    k0 += KS;
    if (DX && k0 >= K) k0 = 0, ++term;
  };
  f32x16 acc[NV][TT];   // [feature block][token block]
#pragma unroll
  for (int f = 0; f < NV; ++f)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[f][t] = f32x16{};
  f32x16 sum[F32 ? NV : 1][F32 ? TT : 1] = {};   // fp32: the folded values of acc
  const int end0 = DX ? a.p[0].k / KS : stages, end1 = DX && a.n > 1 ? end0 + a.p[1].k / KS : stages;   // of the terms
  int fold_at = min(end0, kFold);
  auto fold = [&](int done) {   // after the products of that many stages; the last of them are added below
    if (done != fold_at || done == stages) return;
    fold_at = min(done + kFold, done < end0 ? end0 : done < end1 ? end1 : stages);
#pragma unroll
    for (int f = 0; f < NV; ++f)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        mfma_settled(acc[f][t]);
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[f][t][e] += acc[f][t][e];
        acc[f][t] = f32x16{};
      }
  };
  auto multiply = [&](int buf, int stage) {
    const char* bx = lds + buf * kBuf;
    const char* bw = bx + RA::kBytes;
    if constexpr (!F32) {
      bf16x8 x[2][TT], w[2][NV];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
          x[s][t] = *reinterpret_cast<const bf16x8*>(RA::chunk(bx, wt + 32 * t + col, 2 * s + half));
#pragma unroll
        for (int f = 0; f < NV; ++f) {
          if constexpr (DX) w[s][f] = RT::operand(bw, wf + 32 * f, s, lane);
          else w[s][f] = *reinterpret_cast<const bf16x8*>(RW::chunk(bw, wf + 32 * f + col, 2 * s + half));
        }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int f = 0; f < NV; ++f)
#pragma unroll
          for (int t = 0; t < TT; ++t) acc[f][t] = mfma32(w[s][f], x[s][t], acc[f][t]);
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        f32x4 x[TT], w[NV];   // contraction values 8 s + 4 half + j
#pragma unroll
        for (int t = 0; t < TT; ++t)
          x[t] = *reinterpret_cast<const f32x4*>(RA::chunk(bx, wt + 32 * t + col, 2 * s + half));
#pragma unroll
        for (int f = 0; f < NV; ++f) {
          if constexpr (DX) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              w[f][j] = reinterpret_cast<const float*>(bw)[(8 * s + 4 * half + j) * kFeat + wf + 32 * f + col];
          } else {
            w[f] = *reinterpret_cast<const f32x4*>(RW::chunk(bw, wf + 32 * f + col, 2 * s + half));
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int f = 0; f < NV; ++f)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[f][t] = mfma32x2(w[f][j], x[t][j], acc[f][t]);
      }
      fold(stage + 1);
    }
  };
  auto run = [&](auto use) {
    load(0);
    if (stages > 1) load(1);
    for (int s0 = 0; s0 < stages; s0 += kGemmStages) {
#pragma unroll
      for (int buf = 0; buf < kGemmStages; ++buf) {
        const int s = s0 + buf;
        if (s >= stages) break;
        if (s + 1 < stages) wait_vmcnt<RA::kLoads + kWLoads>();   // this wave's loads of stage s have landed
        else wait_vmcnt<0>();
        __syncthreads();   // every wave's have, and every wave is done with stage s - 1, whose buffer is loaded next
        if (s + 2 < stages) load((buf + 2) % kGemmStages);
        use(buf, s);
      }
    }
  };
  if (live) run(multiply);
  else run([](int, int) {});
  if constexpr (F32) {
#pragma unroll
    for (int f = 0; f < NV; ++f)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        mfma_settled(acc[f][t]);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[f][t][e] += sum[f][t][e];
      }
  }

  const GemmPart& out = a.p[part];
  constexpr bool kHasY = EPI == kPlain || EPI == kMish || EPI == kMab || EPI == kMabResidual;
  constexpr bool kHasOther = EPI == kMab || EPI == kMabResidual || EPI == kDxBase || EPI == kDxMish;
  constexpr bool kHasRes = EPI == kMabResidual || EPI == kAdd;   // the result is fp32
  const T* bias = DX ? nullptr : (const T*)out.bias;
  const T* other = (const T*)a.other;
  T* y = kHasY ? (T*)out.y : nullptr;
  __syncthreads();   // every wave is done with the stage buffers
  if (!live) return;
  char* tile = lds + wave * kWaveOut;   // [32 tokens][32 NV features] fp32, 16-byte slots xor'ed with the token
  constexpr int kRow = 128 * NV, kXor = NV == 1 ? 7 : 15, kLanes = 4 * NV, kPass = 64 / kLanes;   // bytes per row, lanes and tokens per pass
  const int fl = 8 * (lane % kLanes), c = f0 + wf + fl;   // this lane's eight features of the rows it stores
  const bool wide = c + 8 <= cols;                        // fp32 rows may end after four
#pragma unroll
  for (int t = 0; t < TT; ++t) {
#pragma unroll
    for (int f = 0; f < NV; ++f)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int fe = 32 * f + 8 * q + 4 * half;
        f32x4 v = {acc[f][t][4 * q], acc[f][t][4 * q + 1], acc[f][t][4 * q + 2], acc[f][t][4 * q + 3]};
        if (bias && f0 + wf + fe < cols) v += load4f(bias + f0 + wf + fe);
        *reinterpret_cast<f32x4*>(tile + col * kRow + (((fe >> 2) ^ (col & kXor)) << 4)) = v;
      }
#pragma unroll
    for (int pass = 0; pass < 32 / kPass; ++pass) {
      const int tok = pass * kPass + lane / kLanes, row = wt + 32 * t + tok;
      if (row >= nrows || c >= cols) continue;
      const size_t i = (size_t)(row0 + row) * cols + c;
      f32x4 v[2], ov[2] = {}, rv[2] = {}, zv[2];
      if constexpr (kHasOther) load8f(ov, other + i, wide);
      if constexpr (kHasRes) load8f(rv, a.residual + i, wide);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v[h] = *reinterpret_cast<const f32x4*>(tile + tok * kRow + ((((fl >> 2) + h) ^ (tok & kXor)) << 4));
        if constexpr (EPI == kDxBase) v[h] += ov[h];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float z = 0.f;
          v[h][e] = finish<T, EPI>(v[h][e], ov[h][e], rv[h][e], z);
          zv[h][e] = z;
        }
      }
      if constexpr (EPI == kPlain) store8f(y + i, v, wide);
      else {
        if (kHasY && y) store8f(y + i, zv, wide);
        if constexpr (kHasRes) store8f((float*)a.result + i, v, wide);
        else store8f((T*)a.result + i, v, wide);
      }
    }
  }
}

bool gemm_misaligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; }

// The block's tile, 64 tt tokens x 64 nv features.  64 x 64 where larger tiles
// would leave the chip's 256 CUs short of blocks, and for fp32, whose products
// the matrix rate bounds at any tile (33,000 rows, 256 -> 256 features: bf16
// 13.6 vs 15.1 us, fp32 44 vs 56 us; 21,752 x 128 -> 128 fp32 12.5 vs 17.1 us);
// 128 x 256 for long contractions of many blocks, where the LDS reads bound it
// and a wider wave tile needs a quarter fewer (129,850 rows, 2048 -> 512: 321
// vs 358 us; 33,000 rows, 1024 -> 256: 37.7 vs 34.5 us).
struct GemmTile { int tt, nv; };
GemmTile gemm_tile(int64_t rows, int64_t cols, int64_t k, int dtype) {
  const int64_t blocks = (rows + 127) / 128 * ((cols + 127) / 128);   // of 128 x 128
  if (dtype == ESA_F32 || blocks < 768) return GemmTile{1, 1};
  return cols % 256 == 0 && k >= 1024 && blocks >= 2048 ? GemmTile{2, 4} : GemmTile{2, 2};
}

template <int EPI>
int gemm_launch(int dtype, GemmTile t, long long items, hipStream_t st, const GemmArgs& a) {
  if (items > 0x7fffffffLL) return ESA_ERR_SHAPE;
#define ESA_GEMM(T, TT, NV) \
  hipLaunchKernelGGL((linear_gemm_kernel<T, TT, NV, EPI>), dim3((unsigned)items), dim3(256), 0, st, a)
  ESA_TIMED(esa_profile::kLinearGemm, st, {
    if (dtype == ESA_F32) ESA_GEMM(float, 1, 1);
    else if (t.tt == 1) ESA_GEMM(bf16, 1, 1);
    else if (t.nv == 2) ESA_GEMM(bf16, 2, 2);
    else ESA_GEMM(bf16, 2, 4);
  });
#undef ESA_GEMM
  ESA_LAUNCH_CHECK();
  return ESA_OK;
}

// Contraction lengths in whole stages, result widths in 16-byte chunks, rows whose buffer offsets fit.
bool gemm_k_ok(int k, int dtype) { return k >= 32 && k % 32 == 0 && k <= 16384 && (dtype == ESA_F32 || dtype == ESA_BF16); }
bool gemm_cols_ok(int c, int dtype) { return c >= 8 && c % (dtype == ESA_BF16 ? 8 : 4) == 0 && c <= 16384; }

}  // namespace

extern "C" {

int esa_linear_fwd(const void* x, long long rows, int in_features, int dtype, int n, const void* const* weight,
                   const void* const* bias, void* const* y, const int* out_features, int epilogue, const void* other,
                   const float* residual, void* result, void* stream) {
  if (n < 1 || n > kGemmMax || rows < 0 || rows > 0x7fffffff) return ESA_ERR_SHAPE;
  if (dtype != ESA_F32 && dtype != ESA_BF16) return ESA_ERR_DTYPE;
  if (!weight || !bias || !y || !out_features) return ESA_ERR_NULL;
  if (epilogue < ESA_LINEAR_PLAIN || epilogue > ESA_LINEAR_ADD || (epilogue != ESA_LINEAR_PLAIN && n != 1) ||
      !gemm_k_ok(in_features, dtype))
    return ESA_ERR_SHAPE;
  for (int i = 0; i < n; ++i)
    if (!gemm_cols_ok(out_features[i], dtype)) return ESA_ERR_SHAPE;
  if (rows == 0) return ESA_OK;
  const bool needs_other = epilogue == ESA_LINEAR_MAB;
  if (!x || (epilogue != ESA_LINEAR_PLAIN && !result) || (needs_other && !other) ||
      (epilogue == ESA_LINEAR_ADD && !residual))
    return ESA_ERR_NULL;
  if (gemm_misaligned(x) || gemm_misaligned(other) || gemm_misaligned(residual) || gemm_misaligned(result))
    return ESA_ERR_ALIGN;
  GemmArgs a{};
  a.rows = (int)rows; a.n = n; a.x = x; a.other = other; a.residual = residual; a.result = result;
  long long total = 0;
  for (int i = 0; i < n; ++i) total += out_features[i];
  GemmTile t = gemm_tile(rows, total, in_features, dtype);
  for (int i = 0; i < n; ++i)
    if (t.nv == 4 && out_features[i] % 256) t.nv = 2;
  for (int i = 0; i < n; ++i) {
    if (!weight[i] || (epilogue == ESA_LINEAR_PLAIN && !y[i])) return ESA_ERR_NULL;
    if (gemm_misaligned(weight[i]) || gemm_misaligned(y[i]) || gemm_misaligned(bias[i])) return ESA_ERR_ALIGN;
    a.p[i] = GemmPart{nullptr, weight[i], bias[i], y[i], in_features, out_features[i], a.col_tiles};
    a.col_tiles += (out_features[i] + 64 * t.nv - 1) / (64 * t.nv);
  }
  const long long items = (rows + 64 * t.tt - 1) / (64 * t.tt) * a.col_tiles;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch (epilogue) {
    case ESA_LINEAR_PLAIN: return gemm_launch<kPlain>(dtype, t, items, st, a);
    case ESA_LINEAR_MISH: return gemm_launch<kMish>(dtype, t, items, st, a);
    case ESA_LINEAR_MAB:
      return residual ? gemm_launch<kMabResidual>(dtype, t, items, st, a) : gemm_launch<kMab>(dtype, t, items, st, a);
    default: return gemm_launch<kAdd>(dtype, t, items, st, a);
  }
}

int esa_linear_dx(const void* const* g, const void* const* weight, int n, long long rows, const int* out_features,
                  int in_features, int dtype, const void* base, const void* mish_z, void* dx, void* stream) {
  if (n < 1 || n > kGemmMax || rows < 0 || rows > 0x7fffffff || (base && mish_z)) return ESA_ERR_SHAPE;
  if (dtype != ESA_F32 && dtype != ESA_BF16) return ESA_ERR_DTYPE;
  if (!g || !weight || !out_features) return ESA_ERR_NULL;
  if (!gemm_cols_ok(in_features, dtype)) return ESA_ERR_SHAPE;
  for (int i = 0; i < n; ++i)
    if (!gemm_k_ok(out_features[i], dtype)) return ESA_ERR_SHAPE;
  if (rows == 0) return ESA_OK;
  if (!dx) return ESA_ERR_NULL;
  if (gemm_misaligned(base) || gemm_misaligned(mish_z) || gemm_misaligned(dx)) return ESA_ERR_ALIGN;
  GemmArgs a{};
  a.rows = (int)rows; a.n = n; a.cols = in_features; a.result = dx;
  a.other = base ? base : mish_z;
  int64_t contraction = 0;
  for (int i = 0; i < n; ++i) contraction += out_features[i];
  const GemmTile t = gemm_tile(rows, in_features, contraction, dtype);
  for (int i = 0; i < n; ++i) {
    if (!g[i] || !weight[i]) return ESA_ERR_NULL;
    if (gemm_misaligned(g[i]) || gemm_misaligned(weight[i])) return ESA_ERR_ALIGN;
    a.p[i] = GemmPart{g[i], weight[i], nullptr, nullptr, out_features[i], 0, 0};
  }
  a.col_tiles = (in_features + 64 * t.nv - 1) / (64 * t.nv);
  const long long items = (rows + 64 * t.tt - 1) / (64 * t.tt) * a.col_tiles;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (base) return gemm_launch<kDxBase>(dtype, t, items, st, a);
  if (mish_z) return gemm_launch<kDxMish>(dtype, t, items, st, a);
  return gemm_launch<kDx>(dtype, t, items, st, a);
}

}  // extern "C"
