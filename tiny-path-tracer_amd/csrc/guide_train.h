// Guiding network kernels: weight packing, inference, the fused
// forward/backward training step (BF16 MFMA, FP32 accumulation) and the
// gradient reduction + Adam update.
//
// Training step (k_guide_train).  Each wave works on 2 groups of 16 samples at
// a time (lane l: sample l%16 of each group, lane group g = l/16):
//   1. forward in the inference layout (16x16x32, permuted K order, guide.h):
//      the D tiles, "sample-major" (a lane holds neurons 16mt + 4g + r of one
//      sample), feed the next layer directly.  The output rows are permuted so
//      that lane group g holds lobes 2g and 2g+1 of its sample;
//   2. the loss gradient: each lane evaluates its two lobes; the softmax and
//      the mixture density are completed across the sample's four lanes by
//      shuffles, so all 64 lanes work;
//   3. backward data, sample-major, through W4ᵀ, W3ᵀ and W2ᵀ (transposed tiles
//      in the same permuted layout) to chain the deltas; the bias gradients are
//      the lanes' own sums of them;
//   4. dW += δ·hᵀ with v_mfma_f32_16x16x32_bf16, K = the wave's 32 samples.  Its
//      operands are "neuron-major" (a lane holds one neuron of 8 samples): each
//      wave publishes a layer's deltas and activations in LDS, one row of 64
//      neurons per sample, and ds_read_b64_tr_b16 reads 4 samples of a neuron
//      per lane from them.  The 56 dW tiles are split over the block's 8 waves
//      (7 each), every wave adding the products of all 8 waves' samples into
//      the tiles it owns: 28 accumulator registers per wave instead of 224 let
//      two waves share each SIMD (512-thread blocks, one 54 KB copy of the
//      weight tiles per CU).
// Each wave then writes its own tiles into the block partial (every tile has
// one owner); k_guide_finish adds the partials and turns the sum into the
// gradient or the Adam update and the new weight tiles.
#ifndef TPT_CSRC_GUIDE_TRAIN_H
#define TPT_CSRC_GUIDE_TRAIN_H

#include "guide.h"

namespace tptd {

constexpr int G_PARTIAL = G_NPARAM_PAD + 4;  // + mix-logit gradient, loss sum, 2 pad
// Training tile set (1 KB tiles, 16x16x32 layout): forward W1..W4 (W4 rows in
// lobe order), then transposed W4ᵀ, W3ᵀ, W2ᵀ.
constexpr int GR_FWD = 30, GR_BWD = 24, GR_TILES = GR_FWD + GR_BWD;
constexpr int GR_BWD_BASE = GR_FWD;  // W4ᵀ, then W3ᵀ, then W2ᵀ: 8 tiles each

// Output row order of the training forward: physical row p = 16 mt + 4 g + r
// holds output u = 4 mt + r (u < 10) of lane group g, i.e. logical output
// 10 g + u (lobes 2g, 2g+1); rows with u >= 10 are padding.
__host__ __device__ inline int out_phys(int o) {
  const int g = o / 10, u = o % 10;
  return 16 * (u / 4) + 4 * g + (u % 4);
}
__host__ __device__ inline int out_logical(int p) {
  const int u = 4 * (p / 16) + (p % 4);
  return u < 10 ? 10 * ((p % 16) / 4) + u : -1;
}

// Layer geometry: fp32 offset, rows (out), padded cols (in).
__host__ __device__ inline void layer_geom(int L, int *off, int *rows, int *cols) {
  const int o[4] = {G_W1, G_W2, G_W3, G_W4}, r[4] = {64, 64, 64, 48}, c[4] = {48, 64, 64, 64};
  *off = o[L], *rows = r[L], *cols = c[L];
}

// True where a padded-layout parameter is real (not padding).
__host__ __device__ inline bool param_live(int p) {
  if (p < G_W2) return (p % 48) < G_IN;               // W1 cols 42..47 are padding
  if (p < G_W4) return true;
  if (p < G_B1) return (p - G_W4) / 64 < G_OUT;       // W4 rows 40..47
  if (p < G_B4) return true;
  if (p < G_NPARAM_PAD) return (p - G_B4) < G_OUT;    // b4 40..47
  return true;
}

// K slot (s, g, q) of a 16x16x32 operand that holds hidden/output neuron n in
// the permuted order n = 16 (2 s + q/4) + 4 g + q%4 (a lane's own D tiles).
__host__ __device__ inline void neuron_kslot(int n, int *s, int *g, int *q) {
  const int mt = n / 16;
  *s = mt / 2, *g = (n % 16) / 4, *q = 4 * (mt % 2) + (n % 4);
}

// bf16 tile entries of weight t (< G_B1, live) of value w: the inference tiles
// (natural output order) and the training tiles.
__device__ __forceinline__ void guide_pack_weight(int t, float w, uint16_t *__restrict__ xtiles,
                                                  uint16_t *__restrict__ rtiles) {
  const int L = t < G_W2 ? 0 : (t < G_W3 ? 1 : (t < G_W4 ? 2 : 3));
  int off, rows, cols;
  layer_geom(L, &off, &rows, &cols);
  const int o = (t - off) / cols, i = (t - off) % cols;
  const uint16_t v = to_bf16(w);
  // input column i -> K slot
  int g, s, q;
  if (L == 0) {
    int slot;
    feature_xslot(i, &g, &slot);
    s = slot / 8, q = slot % 8;
  } else {
    neuron_kslot(i, &s, &g, &q);
  }
  // inference: natural output rows
  xtiles[((GX_BASE[L] + (o / 16) * 2 + s) * 64 + (o % 16) + 16 * g) * 8 + q] = v;
  // training forward: W4 rows in lobe order
  const int p = L == 3 ? out_phys(o) : o;
  rtiles[((GX_BASE[L] + (p / 16) * 2 + s) * 64 + (p % 16) + 16 * g) * 8 + q] = v;
  // training transposed (A = Wᵀ: rows = inputs i, K = outputs p in the permuted order)
  if (L >= 1) {
    int ks, kg, kq;
    neuron_kslot(p, &ks, &kg, &kq);
    const int tb = GR_BWD_BASE + 8 * (3 - L);  // W4ᵀ at 0, W3ᵀ at 8, W2ᵀ at 16
    rtiles[((tb + (i / 16) * 2 + ks) * 64 + (i % 16) + 16 * kg) * 8 + kq] = v;
  }
}

// All tiles from the fp32 master weights, one thread per (layer, out, in).
// Slots that hold no weight are never written (they stay zero).
__global__ void k_guide_pack(const float *__restrict__ w, uint16_t *__restrict__ xtiles, uint16_t *__restrict__ rtiles) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < G_B1 && param_live(t)) guide_pack_weight(t, w[t], xtiles, rtiles);
}

// (words a multiple of 4; both arrays 16-byte aligned)
// Every load is requested before the first store waits for one.
template <int THREADS, int TILES>
__device__ __forceinline__ void guide_stage_weights(uint32_t *dst, const uint32_t *src) {
  constexpr int N = TILES * GX_TILE_WORDS / 4, K = (N + THREADS - 1) / THREADS;
  f32x4 *d = reinterpret_cast<f32x4 *>(dst);
  const f32x4 *s = reinterpret_cast<const f32x4 *>(src);
  f32x4 v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = s[min(k * THREADS + static_cast<int>(threadIdx.x), N - 1)];
#pragma unroll
  for (int k = 0; k < K; ++k) d[min(k * THREADS + static_cast<int>(threadIdx.x), N - 1)] = v[k];
}

// Raw outputs for inputs in9 (n x 9) -> out (n x 40), on the inference tiles.
//
// What bounds it: HBM, 36 B in and 160 B out per input, once the weights come
// from LDS only half as often.  Each wave takes 2 groups of 16 inputs, so a 1 KB
// tile read feeds 32 of them (the reads of one group each took 24 us per 10^6
// inputs); a lane loads only the 1 to 5 features its group encodes, and stores
// its 4 consecutive outputs at once where the row is 16-byte aligned (VEC).
// 10^6 inputs: 139 -> 75 us, 116 -> 58 us (3.4 TB/s) in buffers that stay cached; 73 us with non-temporal stores, whose
// rows of 160 B end inside cache lines; one group per wave or up to 20 blocks
// per CU are within 3%.
constexpr int GI_GROUPS = 2, GI_ROWS = 4 * 16 * GI_GROUPS;  // inputs per block of 4 waves
template <bool VEC>
__global__ void __launch_bounds__(256) k_guide_infer(const uint32_t *__restrict__ xtiles, const float *__restrict__ params,
                                                     const float *__restrict__ in, uint64_t n, float *__restrict__ out) {
  __shared__ __align__(16) uint32_t wt[GX_TILES * GX_TILE_WORDS];
  __shared__ __align__(16) float bias[G_BIAS];
  guide_stage_weights<256, GX_TILES>(wt, xtiles);
  for (int i = threadIdx.x; i < G_BIAS; i += blockDim.x) bias[i] = params[G_B1 + i];
  __syncthreads();
  const int l = __lane_id(), wave = threadIdx.x / 64, fg = l >> 4;
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * GI_ROWS; base < n;
       base += static_cast<uint64_t>(gridDim.x) * GI_ROWS) {
    bf16x8 xb[GI_GROUPS][2];
    f32x4 o[GI_GROUPS][3];
#pragma unroll
    for (int g = 0; g < GI_GROUPS; ++g) {
      const uint64_t s = base + (wave * GI_GROUPS + g) * 16 + (l & 15);
      const float *row = in + (s < n ? s : n - 1) * 9;
      const float p = fg < 3 ? row[fg] : 0.0f;
      float nwo[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      if (fg == 0) nwo[0] = row[3], nwo[1] = row[4], nwo[2] = row[5], nwo[3] = row[6];
      if (fg == 1) nwo[4] = row[7], nwo[5] = row[8];
      guide_xfeatures(fg, p, nwo, xb[g]);
    }
    guide_forward_groups<GI_GROUPS>(xb, wt, bias, o);
#pragma unroll
    for (int g = 0; g < GI_GROUPS; ++g) {
      const uint64_t s = base + (wave * GI_GROUPS + g) * 16 + (l & 15);
      if (s >= n) continue;
      float *row = out + s * G_OUT;
#pragma unroll
      for (int mt = 0; mt < 3; ++mt) {
        const int f = 16 * mt + 4 * fg;
        if (f >= G_OUT) continue;
        if (VEC) {
          *reinterpret_cast<f32x4 *>(row + f) = o[g][mt];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) row[f + r] = o[g][mt][r];
        }
      }
    }
  }
}

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// One lobe of a sample's mixture, as held by the lane that owns it.
struct lobe {
  float mu[3], nrm, kap, lk, cs, d, w;
};

// raw = (mx, my, mz, log κ); om = the sampled direction ω.
__device__ __forceinline__ void lobe_eval(float a, float b, float c, float lk, v3 om, lobe *L) {
  const float n2 = a * a + b * b + c * c;
  L->nrm = sqrtf(n2);
  if (n2 > 1e-20f) {
    const float inv = rsqrtf(n2);
    L->mu[0] = a * inv, L->mu[1] = b * inv, L->mu[2] = c * inv;
  } else {
    L->mu[0] = 0.0f, L->mu[1] = 0.0f, L->mu[2] = 1.0f;
  }
  L->lk = lk;
  L->kap = __expf(fminf(fmaxf(lk, G_LOGK_MIN), G_LOGK_MAX));
  L->cs = L->mu[0] * om.x + L->mu[1] * om.y + L->mu[2] * om.z;
  L->d = vmf_pdf(L->kap, L->cs);
}

// The lobe's 5 output gradients of -(c/n) log g, given f = -c / (n g) and g.
__device__ __forceinline__ void lobe_grad(const lobe &L, v3 om, float f, float g, float *o5) {
  const float wd = L.w * L.d;
  // d/d raw mean: κ (ω − (μ·ω) μ) / |raw|
  const float s = L.nrm > 1e-10f ? __fdividef(f * wd * L.kap, L.nrm) : 0.0f;
  o5[0] = s * (om.x - L.cs * L.mu[0]);
  o5[1] = s * (om.y - L.cs * L.mu[1]);
  o5[2] = s * (om.z - L.cs * L.mu[2]);
  // d/d log κ: 1 − 2κ/(e^{2κ} − 1) + κ(μ·ω − 1), zero where the clamp is active
  // (2κ ≥ 0.0996: e^{2κ} − 1 ≥ 0.105 keeps ~6 digits; e^{2κ} = inf gives 0)
  const bool live = L.lk > G_LOGK_MIN && L.lk < G_LOGK_MAX;
  o5[3] = live ? f * wd * (1.0f - __fdividef(2.0f * L.kap, __expf(2.0f * L.kap) - 1.0f) + L.kap * (L.cs - 1.0f))
               : 0.0f;
  // d/d logit: w_i (D_i − g)
  o5[4] = f * L.w * (L.d - g);
}

// Block of the training step: 8 waves of 2 groups, 256 samples per iteration.
constexpr int GT_WAVES = 8, GT_GROUPS = 2, GT_SAMPLES = 16 * GT_GROUPS;
constexpr int GT_THREADS = 64 * GT_WAVES, GT_ROWS = GT_SAMPLES * GT_WAVES;
// dW exchange: per wave a delta and an activation row per sample, 64 bf16 each
// in 4 chunks (the tiles) of 4 quads.  Chunk t of row r is stored at t ^ (r/2)%4
// and its quad q at q ^ 2 (r/8 % 2): the 8 rows that half a wave reads one chunk
// of then lie in different banks, and so do the quads of 16 rows that it writes.
constexpr int GT_XROW = 64, GT_XOP = GT_SAMPLES * GT_XROW, GT_XCH = GT_WAVES * 2 * GT_XOP;  // in bf16
constexpr int GT_IROW = 20, GT_IN = GT_WAVES * GT_SAMPLES * GT_IROW;  // staged input rows, in floats
constexpr int GT_SUMS = G_BIAS + 2;  // biases, mix-logit gradient, loss

constexpr size_t k_guide_train_lds() { return GR_TILES * 1024 + G_BIAS * 4 + GT_XCH * 2 + GT_IN * 4; }
static_assert(GT_WAVES * GT_SUMS * 4 <= GT_XCH * 2, "the waves' sums take the exchange's place");
static_assert(k_guide_train_lds() <= 160 * 1024, "one block per CU");

// dW tile (mo, ni) of weight layer L owned by wave w in slot e (0, 1): the two
// share an operand.  The first layer's second slot goes to the waves whose
// second slot is empty in the last one, so that each wave owns 7.  False if the
// slot holds no tile.
__device__ __forceinline__ bool owned_tile(int w, int L, int e, int *mo, int *ni) {
  if (L == 0) {
    *mo = w % 4, *ni = w / 4 + e;
    return e == 0 || w >= 4;
  }
  *mo = w / 4 + 2 * e, *ni = w % 4;
  return L < 3 || *mo < 3;
}

// 8 samples of neuron (l % 16) of a tile: lane addresses from `at` (this lane's
// 4 neurons of sample 4 (l / 16) + (l % 16) / 4), groups 0 and 1.
__device__ __forceinline__ bf16x8 read_neurons(const uint16_t *at) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 *lds_ptr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(const_cast<uint16_t *>(at)));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(const_cast<uint16_t *>(at + 16 * GT_XROW)));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Sum over the 16 lanes of a row, in every lane (rotations by 8, 4, 2, 1).
__device__ __forceinline__ float row_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xF, 0xF, true));
  return v;
}

// Sums of 16 values over the 16 lanes of a row, value j in lane j (j = l % 16):
// each step adds the half of the values that the partner lane keeps.
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ float row_scatter(f32x16 v, int j) {
#pragma unroll
  for (int w = 8; w > 0; w /= 2) {
    const bool hi = (j & w) != 0;
#pragma unroll
    for (int k = 0; k < w; ++k) {
      const float a = v[k], b = v[k + w], keep = hi ? b : a, give = hi ? a : b;
      const int x = __float_as_int(give);
      // partners: lane 15 - j, 7 - j within 8, j ^ 2, j ^ 1
      const int y = w == 8   ? __builtin_amdgcn_update_dpp(0, x, 0x140, 0xF, 0xF, true)
                    : w == 4 ? __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, true)
                    : w == 2 ? __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, true)
                             : __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true);
      v[k] = keep + __int_as_float(y);
    }
  }
  return v[0];
}

// v gated by ReLU' of the activations a (bf16, >= 0): element 4 (mt % 2) + r of
// a[mt / 2] belongs to v[r].
__device__ __forceinline__ f32x4 relu_gate(f32x4 v, const bf16x8 a[2], int mt) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 w = __builtin_bit_cast(u32x4, a[mt / 2]);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t x = w[2 * (mt % 2) + k];
    v[2 * k] = (x & 0xFFFFu) ? v[2 * k] : 0.0f;
    v[2 * k + 1] = x > 0xFFFFu ? v[2 * k + 1] : 0.0f;
  }
  return v;
}

// What bounds it: two waves per SIMD in step with each other, each waiting on
// LDS and on chains of dependent products (LDS 35%, vector ALU 42%, matrix cores
// 14% busy).  So a wave takes two groups of samples, each weight tile read from
// LDS serves both and the products of one fill the gaps of the other; the
// neuron-major operands come from a transposing LDS read of what the forward
// pass holds anyway (computing them again with swapped operands and identity
// tiles took as many products and tile reads as all the rest); the bias sums
// live in 4 registers (60 without row_scatter, and 60 spilled); the next rows
// are requested an iteration ahead.  2^18 rows: 105.6 -> 57 us, a step with
// k_guide_finish 122 -> 67 us; 4096 rows: a step 37.8 -> 25.2 us.  The bias is
// added after the products (inside them it rounds differently, and Adam's
// division by the gradient's own size makes 2e-3 of that after 8 steps).
//
// Fused forward/backward over rows [0, n) (row k read at (row0 + k) % n_total;
// row0 < n_total, n <= n_total).  GT_THREADS threads per block; each wave takes
// 32 rows, the block 256 per iteration.  Writes this block's partial gradient
// (natural parameter layout) to partial.
__global__ void __launch_bounds__(GT_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
k_guide_train(const uint32_t *__restrict__ rtiles, const float *__restrict__ params, const float *__restrict__ rows,
              uint64_t n, uint64_t row0, uint64_t n_total, float *__restrict__ partial) {
  extern __shared__ __align__(16) uint8_t lds[];
  uint32_t *wt = reinterpret_cast<uint32_t *>(lds);
  float *bias = reinterpret_cast<float *>(wt + GR_TILES * 256);  // b1 b2 b3 natural, b4 in lobe order
  uint16_t *xch = reinterpret_cast<uint16_t *>(bias + G_BIAS);   // dW exchange (GT_XCH)
  float *stage = reinterpret_cast<float *>(xch + GT_XCH);        // input rows (GT_IN)
  const int l = __lane_id(), g = l >> 4, j = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);  // (kept scalar)
  // Rows of the block's next iteration, requested an iteration ahead: lane l
  // holds 16 bytes of rows l/4 and 16 + l/4 (4-byte aligned as the caller's are).
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 nxt[GT_GROUPS];
  const auto request = [&](uint64_t bbase) {
#pragma unroll
    for (int k = 0; k < GT_GROUPS; ++k) {
      const uint64_t at = bbase + GT_SAMPLES * wave + 16 * k + l / 4;
      nxt[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (at < n) {
        uint64_t r = row0 + at;
        r = r >= n_total ? r - n_total : r;
        nxt[k] = *reinterpret_cast<const f32x4u *>(rows + r * TPT_GUIDE_ROW + 4 * (l % 4));
      }
    }
  };
  request(static_cast<uint64_t>(blockIdx.x) * GT_ROWS);
  guide_stage_weights<GT_THREADS, GR_TILES>(wt, rtiles);
  for (int i = threadIdx.x; i < G_BIAS; i += blockDim.x) {
    float b = 0.0f;
    if (i < 192) b = params[G_B1 + i];
    else if (out_logical(i - 192) >= 0) b = params[G_B4 + out_logical(i - 192)];
    bias[i] = b;
  }
  __syncthreads();
  const bf16x8 *T = reinterpret_cast<const bf16x8 *>(wt);
  const f32x4 *bias4 = reinterpret_cast<const f32x4 *>(bias);  // bias4[4 t + g]: rows 16 t + 4 g .. + 3
  const float inv_n = 1.0f / static_cast<float>(n);
  const float alpha = 1.0f / (1.0f + __expf(-params[G_NPARAM_PAD]));
  // the dW tiles this wave owns, slot 2 L + e (owned_tile), accumulated over the launch
  f32x4 dw[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) dw[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float db[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // bias gradient of neuron 16 (j / 4) + 4 g + j % 4 of each layer
  float dalpha = 0.0f, loss = 0.0f;
  float *in_w = stage + wave * GT_SAMPLES * GT_IROW;
  uint16_t *xw = xch + wave * 2 * GT_XOP + j * GT_XROW;  // this lane's sample row of group 0
  const int wc = (j / 2) % 4, wq = 2 * (j / 8);          // its chunk and quad swizzles
  const int rrow = 4 * g + j / 4, rc = (rrow / 2) % 4;
  const uint16_t *xr = xch + rrow * GT_XROW + 4 * ((j % 4) ^ (2 * (rrow / 8)));  // read_neurons: wave 0
  // every wave of a block runs the same iterations (the dW exchange has block
  // barriers); a wave past the end works on zero-weight rows
  for (uint64_t bbase = static_cast<uint64_t>(blockIdx.x) * GT_ROWS; bbase < n;
       bbase += static_cast<uint64_t>(gridDim.x) * GT_ROWS) {
    // an opaque zero offset keeps the weight-tile loads inside the loop (hoisted
    // out of it they would hold the whole tile set in registers)
    int zoff = 0;
    asm volatile("" : "+v"(zoff));
    const bf16x8 *Tl = T + zoff + l;
    const f32x4 *bl = bias4 + zoff + g;
#pragma unroll
    for (int k = 0; k < GT_GROUPS; ++k)
      *reinterpret_cast<f32x4 *>(in_w + (16 * k + l / 4) * GT_IROW + 4 * (l % 4)) = nxt[k];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    request(bbase + static_cast<uint64_t>(gridDim.x) * GT_ROWS);
    __syncthreads();  // every wave has read the exchange of the iteration before
    // ---- 1. forward, sample-major.  The wave's exchange rows are its own until
    // the first delta is published and keep the first two layers' inputs.
    bf16x8 xa[GT_GROUPS][2], a1[GT_GROUPS][2], a2[GT_GROUPS][2], a3[GT_GROUPS][2];
#pragma unroll
    for (int k = 0; k < GT_GROUPS; ++k) {
      const float *r = in_w + (16 * k + j) * GT_IROW;
      const f32x4 r4 = *reinterpret_cast<const f32x4 *>(r + 4);
      const float nwo[6] = {r[3], r4[0], r4[1], r4[2], r4[3], r[8]};
      guide_xfeatures(g, r[g < 3 ? g : 2], nwo, xa[k]);
    }
#pragma unroll
    for (int layer = 0; layer < 3; ++layer) {
      f32x4 acc[GT_GROUPS][4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int k = 0; k < GT_GROUPS; ++k) acc[k][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const bf16x8 w = Tl[(GX_BASE[layer] + 2 * mt + s) * 64];
#pragma unroll
          for (int k = 0; k < GT_GROUPS; ++k)
            acc[k][mt] = mfma32(w, layer == 0 ? xa[k][s] : (layer == 1 ? a1[k][s] : a2[k][s]), acc[k][mt]);
        }
      }
#pragma unroll
      for (int k = 0; k < GT_GROUPS; ++k) {
        // (the larger of z and 0, 0 for a NaN)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          const f32x4 b = bl[4 * (4 * layer + mt)];
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[k][mt][r] = fmaxf(acc[k][mt][r] + b[r], 0.0f);
        }
        bf16x8 *out = layer == 0 ? a1[k] : (layer == 1 ? a2[k] : a3[k]);
        out[0] = pack8(acc[k][0], acc[k][1]);
        out[1] = pack8(acc[k][2], acc[k][3]);
        if (layer < 2) {
          bf16x8 *keep = reinterpret_cast<bf16x8 *>(xw + (16 * k) * GT_XROW + layer * GT_XOP + 16 * (g ^ wc));
          keep[0] = layer == 0 ? xa[k][0] : a1[k][0];
          keep[1] = layer == 0 ? xa[k][1] : a1[k][1];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x4 o[GT_GROUPS][3];
#pragma unroll
    for (int mt = 0; mt < 3; ++mt) {
#pragma unroll
      for (int k = 0; k < GT_GROUPS; ++k) o[k][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 w = Tl[(GX_BASE[3] + 2 * mt + s) * 64];
#pragma unroll
        for (int k = 0; k < GT_GROUPS; ++k) o[k][mt] = mfma32(w, a3[k][s], o[k][mt]);
      }
      const f32x4 b = bl[4 * (12 + mt)];
#pragma unroll
      for (int k = 0; k < GT_GROUPS; ++k) o[k][mt] += b;
    }
    // ---- 2. loss gradient: this lane holds lobes 2g (o0.xyzw, o1.x) and 2g+1 (o1.yzw, o2.xy)
    bf16x8 dup[GT_GROUPS][2];  // the current layer's output delta, sample-major
    f32x16 dsum = {};
#pragma unroll
    for (int k = 0; k < GT_GROUPS; ++k) {
      const float *r = in_w + (16 * k + j) * GT_IROW;
      const v3 om{r[9], r[10], r[11]};
      const float c = r[12], qd = r[13];
      const bool use = c > 0.0f && c < 3.0e38f;  // (rows past the end are zeros)
      lobe A, B;
      lobe_eval(o[k][0][0], o[k][0][1], o[k][0][2], o[k][0][3], om, &A);
      lobe_eval(o[k][1][1], o[k][1][2], o[k][1][3], o[k][2][0], om, &B);
      const float la = o[k][1][0], lb = o[k][2][1];
      float mx = fmaxf(la, lb);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float ea = __expf(la - mx), eb = __expf(lb - mx);
      float z = ea + eb;
      z += __shfl_xor(z, 16);
      z += __shfl_xor(z, 32);
      const float iz = __fdividef(1.0f, z);
      A.w = ea * iz, B.w = eb * iz;
      float gp = A.w * A.d + B.w * B.d;
      gp += __shfl_xor(gp, 16);
      gp += __shfl_xor(gp, 32);
      gp = fmaxf(gp, 1e-30f);
      const float f = use ? __fdividef(-c * inv_n, gp) : 0.0f;
      float ga[5], gb[5];
      lobe_grad(A, om, f, gp, ga);
      lobe_grad(B, om, f, gp, gb);
      f32x4 d[3];
      d[0] = use ? f32x4{ga[0], ga[1], ga[2], ga[3]} : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      d[1] = use ? f32x4{ga[4], gb[0], gb[1], gb[2]} : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      d[2] = use ? f32x4{gb[3], gb[4], 0.0f, 0.0f} : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (use && g == 0) {
        loss += -c * __logf(gp);
        const float mm = alpha * gp + (1.0f - alpha) * qd;
        if (mm > 0.0f) dalpha += __fdividef(-c * inv_n * (gp - qd) * alpha * (1.0f - alpha), mm);
      }
      dup[k][0] = pack8(d[0], d[1]);
      dup[k][1] = pack8(d[2], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
      // (the output biases take the delta as the weights do: rounded)
#pragma unroll
      for (int u = 0; u < 10; ++u) dsum[u] += static_cast<float>(dup[k][u / 8][u % 8]);
    }
    db[3] += row_scatter(dsum, j);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < GT_GROUPS; ++k) {
      const bf16x8 *keep = reinterpret_cast<const bf16x8 *>(xw + (16 * k) * GT_XROW + 16 * (g ^ wc));
      xa[k][0] = keep[0], xa[k][1] = keep[1];
      a1[k][0] = keep[GT_XOP / 8], a1[k][1] = keep[GT_XOP / 8 + 1];
    }
    // ---- 3, 4. layer by layer from the top: publish δ_L and its input
    // activations, add every wave's δ hᵀ into the owned tiles, next delta.
#pragma unroll
    for (int L = 3; L >= 0; --L) {
      if (L < 3) __syncthreads();  // every wave has read the layer before
#pragma unroll
      for (int k = 0; k < GT_GROUPS; ++k) {
        uint16_t *dl = xw + 16 * k * GT_XROW, *hl = dl + GT_XOP;
        const bf16x8 *h = L == 3 ? a3[k] : (L == 2 ? a2[k] : (L == 1 ? a1[k] : xa[k]));
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          const u32x4 dv = __builtin_bit_cast(u32x4, dup[k][mt / 2]), hv = __builtin_bit_cast(u32x4, h[mt / 2]);
          const int e = 2 * (mt % 2);
          const int at = 16 * (mt ^ wc) + 4 * (g ^ wq);
          if (L < 3 || mt < 3) *reinterpret_cast<u32x2 *>(dl + at) = u32x2{dv[e], dv[e + 1]};
          if (L > 0) *reinterpret_cast<u32x2 *>(hl + at) = u32x2{hv[e], hv[e + 1]};
        }
        if (L == 0) {  // input slots 16 g + t (the last group holds none)
          *reinterpret_cast<bf16x8 *>(hl + 16 * (g ^ wc) + 4 * wq) = h[0];
          *reinterpret_cast<bf16x8 *>(hl + 16 * (g ^ wc) + 8 - 4 * wq) = h[1];
        }
      }
      __syncthreads();
      int mo[2], ni[2];
      (void)owned_tile(wave, L, 0, &mo[0], &ni[0]);
      const bool two = owned_tile(wave, L, 1, &mo[1], &ni[1]);
      const uint16_t *xd = xr + 16 * (mo[0] ^ rc), *xh = xr + GT_XOP + 16 * (ni[0] ^ rc);
      // the second tile's own operand
      const uint16_t *x2 = L == 0 ? xr + GT_XOP + 16 * (ni[1] ^ rc) : xr + 16 * (mo[1] ^ rc);
      if (two) {
#pragma unroll
        for (int src = 0; src < GT_WAVES; ++src) {
          const int at = src * 2 * GT_XOP;
          const bf16x8 a = read_neurons(xd + at), b = read_neurons(xh + at);
          dw[2 * L] = mfma32(a, b, dw[2 * L]);
          const bf16x8 c = read_neurons(x2 + at);
          dw[2 * L + 1] = L == 0 ? mfma32(a, c, dw[2 * L + 1]) : mfma32(c, b, dw[2 * L + 1]);
        }
      } else {
#pragma unroll
        for (int src = 0; src < GT_WAVES; ++src) {
          const int at = src * 2 * GT_XOP;
          dw[2 * L] = mfma32(read_neurons(xd + at), read_neurons(xh + at), dw[2 * L]);
        }
      }
      // δ_{L-1}: (W_Lᵀ δ_L) ⊙ ReLU'
      if (L > 0) {
        f32x4 acc[GT_GROUPS][4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
          for (int k = 0; k < GT_GROUPS; ++k) acc[k][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const bf16x8 w = Tl[(GR_BWD_BASE + 8 * (3 - L) + 2 * mt + s) * 64];
#pragma unroll
            for (int k = 0; k < GT_GROUPS; ++k) acc[k][mt] = mfma32(w, dup[k][s], acc[k][mt]);
          }
        }
#pragma unroll
        for (int k = 0; k < GT_GROUPS; ++k) {
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) {
            acc[k][mt] = relu_gate(acc[k][mt], L == 3 ? a3[k] : (L == 2 ? a2[k] : a1[k]), mt);
#pragma unroll
            for (int r = 0; r < 4; ++r) dsum[4 * mt + r] = k == 0 ? acc[k][mt][r] : dsum[4 * mt + r] + acc[k][mt][r];
          }
          dup[k][0] = pack8(acc[k][0], acc[k][1]);
          dup[k][1] = pack8(acc[k][2], acc[k][3]);
        }
        db[L - 1] += row_scatter(dsum, j);
      }
    }
  }
  // biases, mix logit, loss: in LDS, over the waves in order
  __syncthreads();
  float *sums = reinterpret_cast<float *>(xch);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k < 3 || j < 12) sums[wave * GT_SUMS + 64 * k + 16 * (j / 4) + 4 * g + j % 4] = db[k];
  // (lane group 0 holds them)
  dalpha = row_sum(dalpha);
  loss = row_sum(loss);
  if (l == 0) {
    sums[wave * GT_SUMS + G_BIAS] = dalpha;
    sums[wave * GT_SUMS + G_BIAS + 1] = loss;
  }
  __syncthreads();
  float *P = partial + static_cast<size_t>(blockIdx.x) * G_PARTIAL;
  // this wave's tiles: tile (L, mo, ni), lane (g, j), register r holds
  // dW[16 mo + 4 g + r][column 16 ni + j]
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int L = k / 2;
    int mo, ni;
    if (!owned_tile(wave, L, k % 2, &mo, &ni)) continue;
    int off, rws, cols;
    layer_geom(L, &off, &rws, &cols);
    const int col = L == 0 ? xslot_feature(ni, j) : 16 * ni + j;  // input slot (g, t) at 16 g + t
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rr = 16 * mo + 4 * g + r;
      const int row_ = L == 3 ? out_logical(rr) : rr;
      if (row_ >= 0 && col >= 0) P[off + row_ * cols + col] = dw[k][r];
    }
  }
  for (int i = threadIdx.x; i < GT_SUMS; i += blockDim.x) {
    float v = 0.0f;
    for (int w = 0; w < GT_WAVES; ++w) v += sums[w * GT_SUMS + i];
    if (i >= G_BIAS) P[G_NPARAM_PAD + (i - G_BIAS)] = v;
    else if (i < 192) P[G_B1 + i] = v;
    else if (out_logical(i - 192) >= 0) P[G_B4 + out_logical(i - 192)] = v;
  }
}

// What bounds it: the latency of the partials (15 MB at 256 blocks): 16 loads in
// flight per thread, and no launch after it.  6.5 us in place of the three
// launches of 16 us that added the partials with atomics, stepped and packed.
//
// Sums the block partials (64 parameters x 16 parts per block of 1024) and
// consumes the sum: mode 0 writes the gradient to grad, mode 1 applies Adam
// (step `step`, learning rate lr) and writes the new weight's tile entries.
constexpr int GF_PARAMS = 64, GF_PARTS = 16, GF_THREADS = GF_PARAMS * GF_PARTS;
__global__ void __launch_bounds__(GF_THREADS)
k_guide_finish(const float *__restrict__ partial, int blocks, float *__restrict__ params, float *__restrict__ adam_m,
               float *__restrict__ adam_v, float *__restrict__ grad, float *__restrict__ loss_out, int mode, float lr,
               int step, uint16_t *__restrict__ xtiles, uint16_t *__restrict__ rtiles) {
  __shared__ float part[GF_PARTS][GF_PARAMS];
  const int p = blockIdx.x * GF_PARAMS + threadIdx.x % GF_PARAMS, k = threadIdx.x / GF_PARAMS;
  float s = 0.0f;
  if (p <= G_NPARAM_PAD + 1) {
#pragma unroll 16
    for (int b = k; b < blocks; b += GF_PARTS) s += partial[static_cast<size_t>(b) * G_PARTIAL + p];
  }
  part[k][threadIdx.x % GF_PARAMS] = s;
  __syncthreads();
  if (k > 0 || p > G_NPARAM_PAD + 1) return;
  float g = 0.0f;
  for (int i = 0; i < GF_PARTS; ++i) g += part[i][threadIdx.x];
  if (p == G_NPARAM_PAD + 1) {
    if (loss_out) *loss_out = g;
    return;
  }
  if (!param_live(p)) g = 0.0f;
  if (mode == 0) {
    grad[p] = g;
    return;
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float m = b1 * adam_m[p] + (1.0f - b1) * g;
  const float v = b2 * adam_v[p] + (1.0f - b2) * g * g;
  adam_m[p] = m;
  adam_v[p] = v;
  if (!param_live(p)) return;
  const float mh = m / (1.0f - powf(b1, static_cast<float>(step)));
  const float vh = v / (1.0f - powf(b2, static_cast<float>(step)));
  float w = params[p] - lr * mh / (sqrtf(vh) + eps);
  if (p == G_NPARAM_PAD) w = fminf(fmaxf(w, -3.0f), 3.0f);  // mix weight in [0.05, 0.95]
  params[p] = w;
  if (p < G_B1) guide_pack_weight(p, w, xtiles, rtiles);
}

}  // namespace tptd

#endif  // TPT_CSRC_GUIDE_TRAIN_H
