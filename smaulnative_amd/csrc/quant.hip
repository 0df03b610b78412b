// quant.hip -- the tiled E4M3 quantizer on MI355X (gfx950).
//
// Replaces the reference's native quantizer kernel/quant_cpu.cpp:64-137
// (fp8_quantize_tiles, reached through CpuBackend.fp8_quantize_tiles,
// kernel/compute.py:246-263) and gives the same codes and scales as its torch
// path (kernel/fp8_tile.py:100-113), bit for bit:
//   amax_t = max |w| over the finite entries of the tile, at least 1e-12
//   sc_t   = max(amax_t / 448, 1e-12)
//   n      = clamp(nan_to_num(w / sc_t, nan=0), -448, 448)
//   code   = order[first i with bounds[i] >= n]       (0 where n == 0)
// `order` / `bounds` are the sorted-codebook permutation and its 255
// midpoints, passed in by the caller from the same tables the reference
// uses: the codebook has duplicate values (0x7E/0x7F = 448, 0xFE/0xFF =
// -448), so which duplicate a saturated weight gets is the tables' tie order.
//
// Layout: w fp32 [out_f, in_f] row-major; codes uint8 [out_f, ldc] with
// ldc >= nt * tile (the padding of the last tile is written as code 0, as the
// reference returns it); scales fp32 [out_f, nt].  An HBM-bound pass: 4 bytes
// read and 1 written per weight, every tile read once.
//
// The same rules close the weight update (requant, kernel/fp8_tile.py:240-285):
// w = decode(codes) * scale, times 1 - decay, minus the update (or Lion's,
// whose momentum advances in place), quantized again, in one pass over the
// matrix (QuantSrc).
#include "e4m3.h"
#include "smaul_common.h"

using smaul::check_launch;
using smaul::fail;

namespace {

constexpr int QUANT_THREADS = 256;

__global__ void quant_clear_kernel(unsigned long long* counter) { *counter = 0ull; }

// Where the fp32 weights come from.  QS_MATRIX: w as it is.  QS_REQUANT: the
// decoded codes, decayed, minus `update` (none: null).  QS_LION: the decoded
// codes, decayed, minus sign(b1 m + c1 g) lr, and m advances to b2 m + c2 g.
// Rounded where the reference's tensor operations round: every product and
// sum by itself, but for the momentum's second product, which its add fuses.
enum { QS_MATRIX = 0, QS_REQUANT = 1, QS_LION = 2 };
struct QuantSrc {
  const float* w;
  const uint8_t* codes;
  const float* scales;
  const float* update;
  const void* g;   // fp32 or bf16
  float* m;
  int g_bf16, decay;
  float keep, lr, b1, c1, b2, c2;
};

__device__ __forceinline__ float quant_update(const QuantSrc& p, int mode, float w, float u, float g, float& m) {
  if (p.decay) w = w * p.keep;
  if (mode == QS_LION) {
    const float d = m * p.b1 + g * p.c1;
    u = ((float)(d > 0.0f) - (float)(d < 0.0f)) * p.lr;
    m = __builtin_fmaf(p.c2, g, m * p.b2);
    return w - u;
  }
  return p.update ? w - u : w;
}

// weight (row, k), k < in_f, whose tile has scale index t; LION: writes m when `store`
template <int MODE>
__device__ __forceinline__ float quant_weight(const QuantSrc& p, int64_t row, int64_t k, int64_t in_f, int64_t t,
                                              int64_t nt, bool store) {
  const int64_t e = row * in_f + k;
  if constexpr (MODE == QS_MATRIX) return p.w[e];
  const float w = __builtin_amdgcn_cvt_f32_fp8((int)canon4(p.codes[e]), 0) * p.scales[row * nt + t];
  float g = 0.0f, m = 0.0f, u = 0.0f;
  if constexpr (MODE == QS_LION) {
    g = p.g_bf16 ? bf2f(((const uint16_t*)p.g)[e]) : ((const float*)p.g)[e];
    m = p.m[e];
  } else if (p.update) {
    u = p.update[e];
  }
  const float v = quant_update(p, MODE, w, u, g, m);
  if constexpr (MODE == QS_LION)
    if (store) p.m[e] = m;
  return v;
}

// The scaled weight's code: order[first i in [0, 255] with bounds[i] >= n]
// (std::lower_bound / torch.bucketize), 0 where n is 0.  The search starts
// from the rank of the hardware's nearest code (the sorted codebook holds the
// negatives descending below 128, the others from it), at most a step or two
// away; it ends at the same i from any start.
__device__ __forceinline__ uint32_t quant_encode(float v, float sc, const float* sb, const uint8_t* so) {
  float n = v / sc;
  if (n != n) n = 0.0f;
  if (n == 0.0f) return 0u;  // all of a tile's padding, in wide tiles whole waves of it
  n = fminf(fmaxf(n, -448.0f), 448.0f);
  const int mag = __builtin_amdgcn_cvt_pk_fp8_f32(n, n, 0, false) & 0x7f;
  int r = n < 0.0f ? 127 - mag : 128 + mag;
  while (r > 0 && sb[r - 1] >= n) --r;
  while (r < 255 && sb[r] < n) ++r;
  return so[r];
}

__device__ __forceinline__ float quant_scale(float amax) {
  const float am = amax < 1e-12f ? 1e-12f : amax;
  return fmaxf(am / 448.0f, 1e-12f);
}

// the wave's non-finite count, one atomic per wave that saw any
__device__ __forceinline__ void quant_count(int bad, unsigned long long* nonfinite) {
  for (int o = 32; o >= 1; o >>= 1) bad += __shfl_xor(bad, o, 64);
  if ((threadIdx.x & 63) == 0 && bad) atomicAdd(nonfinite, (unsigned long long)bad);
}

__device__ __forceinline__ void quant_tables(const float* bounds, const uint8_t* order, float* sb, uint8_t* so) {
  if (threadIdx.x < 255) sb[threadIdx.x] = bounds[threadIdx.x];
  if (threadIdx.x < 256) so[threadIdx.x] = order[threadIdx.x];
  __syncthreads();
}

// Four consecutive weights a lane, tile / 4 lanes a tile (tile a power of two
// from 4 to 256), 16-byte rows: the pass streams 12 bytes a weight with Lion, 5
// for a plain matrix.  2560 x 1024: Lion 13.9 us (2.3 TB/s; as a dozen tensor
// operations and the quantizer 85 us), bound by the division and the table
// reads per weight more than by the bytes.  A lane per weight and a binary
// search of eight dependent LDS reads took 24 us for the plain matrix alone.
template <int MODE>
__global__ void __launch_bounds__(QUANT_THREADS)
quant_vec_kernel(QuantSrc p, int64_t out_f, int64_t in_f, int tile, int64_t nt, int64_t ldc,
                 const uint8_t* __restrict__ order, const float* __restrict__ bounds, uint8_t* __restrict__ codes,
                 float* __restrict__ scales, unsigned long long* __restrict__ nonfinite, int64_t units) {
  __shared__ float sb[256];
  __shared__ uint8_t so[256];
  quant_tables(bounds, order, sb, so);
  const int lane = threadIdx.x & 63;
  const int64_t unit = ((int64_t)blockIdx.x * QUANT_THREADS + threadIdx.x) >> 6;
  if (unit >= units) return;  // whole waves: the shuffles below stay uniform
  const int tl = tile >> 2, per_wave = 64 / tl;  // lanes of a tile, tiles of a wave
  const int64_t waves_per_row = (nt + per_wave - 1) / per_wave;
  const int64_t row = unit / waves_per_row;
  const int64_t t = (unit % waves_per_row) * per_wave + lane / tl;
  const int64_t k = t * tile + (lane % tl) * 4;
  const bool in = t < nt && k < in_f;  // in_f % 4 == 0: all four or none
  const int64_t e = row * in_f + k;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (in) {
    if constexpr (MODE == QS_MATRIX) {
      const float4 w = *(const float4*)(p.w + e);
      v[0] = w.x, v[1] = w.y, v[2] = w.z, v[3] = w.w;
    } else {
      const uint32_t c = canon4(*(const uint32_t*)(p.codes + e));
      const float s = p.scales[row * nt + t];
      const float w[4] = {__builtin_amdgcn_cvt_f32_fp8((int)c, 0) * s, __builtin_amdgcn_cvt_f32_fp8((int)c, 1) * s,
                          __builtin_amdgcn_cvt_f32_fp8((int)c, 2) * s, __builtin_amdgcn_cvt_f32_fp8((int)c, 3) * s};
      float u[4] = {0.0f, 0.0f, 0.0f, 0.0f}, g[4] = {0.0f, 0.0f, 0.0f, 0.0f}, m[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if constexpr (MODE == QS_LION) {
        const float4 m4 = *(const float4*)(p.m + e);
        m[0] = m4.x, m[1] = m4.y, m[2] = m4.z, m[3] = m4.w;
        if (p.g_bf16) {
          const uint2 b = *(const uint2*)((const uint16_t*)p.g + e);
          g[0] = bf2f(b.x & 0xffffu), g[1] = bf2f(b.x >> 16), g[2] = bf2f(b.y & 0xffffu), g[3] = bf2f(b.y >> 16);
        } else {
          const float4 g4 = *(const float4*)((const float*)p.g + e);
          g[0] = g4.x, g[1] = g4.y, g[2] = g4.z, g[3] = g4.w;
        }
      } else if (p.update) {
        const float4 u4 = *(const float4*)(p.update + e);
        u[0] = u4.x, u[1] = u4.y, u[2] = u4.z, u[3] = u4.w;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = quant_update(p, MODE, w[q], u[q], g[q], m[q]);
      if constexpr (MODE == QS_LION) *(float4*)(p.m + e) = make_float4(m[0], m[1], m[2], m[3]);
    }
  }
  int bad = 0;
  float amax = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool fin = __builtin_isfinite(v[q]);
    bad += !fin;
    amax = fin ? fmaxf(amax, fabsf(v[q])) : amax;
  }
  for (int o = 1; o < tl; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  const float sc = quant_scale(amax);
  if (t < nt && k < ldc) {
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) c |= quant_encode(v[q], sc, sb, so) << (8 * q);
    *(uint32_t*)(codes + row * ldc + k) = c;
    if (lane % tl == 0) scales[row * nt + t] = sc;
  }
  quant_count(bad, nonfinite);
}

// SEG: tile is a power of two <= 64; a wave covers 64 / tile consecutive
// tiles of one row, lanes in aligned segments of `tile`.  Otherwise a wave
// covers one tile, lane l holding elements l, l + 64, ... of it.
template <int MODE, bool SEG>
__global__ void __launch_bounds__(QUANT_THREADS)
quant_tiles_kernel(QuantSrc p, int64_t out_f, int64_t in_f, int tile, int64_t nt, int64_t ldc,
                   const uint8_t* __restrict__ order, const float* __restrict__ bounds, uint8_t* __restrict__ codes,
                   float* __restrict__ scales, unsigned long long* __restrict__ nonfinite, int64_t units) {
  __shared__ float sb[256];
  __shared__ uint8_t so[256];
  quant_tables(bounds, order, sb, so);
  const int lane = threadIdx.x & 63;
  const int64_t unit = ((int64_t)blockIdx.x * QUANT_THREADS + threadIdx.x) >> 6;
  if (unit >= units) return;  // whole waves: the shuffles below stay uniform
  const int per_wave = SEG ? 64 / tile : 1;            // tiles per wave
  const int64_t waves_per_row = (nt + per_wave - 1) / per_wave;
  const int64_t row = unit / waves_per_row;
  const int64_t t = (unit % waves_per_row) * per_wave + (SEG ? lane / tile : 0);
  int bad = 0;
  float amax = 0.0f;
  if constexpr (SEG) {
    const int64_t k = t * tile + lane % tile;
    float v = 0.0f;
    if (t < nt && k < in_f) v = quant_weight<MODE>(p, row, k, in_f, t, nt, true);
    if (!__builtin_isfinite(v)) ++bad;
    amax = __builtin_isfinite(v) ? fabsf(v) : 0.0f;
    for (int o = 1; o < tile; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    const float sc = quant_scale(amax);
    if (t < nt) {
      if (k < ldc) codes[row * ldc + k] = (uint8_t)quant_encode(v, sc, sb, so);
      if (lane % tile == 0) scales[row * nt + t] = sc;
    }
  } else {
    const int64_t k0 = t * tile;
    for (int j = lane; j < tile; j += 64) {
      const int64_t k = k0 + j;
      const float v = k < in_f ? quant_weight<MODE>(p, row, k, in_f, t, nt, false) : 0.0f;
      if (!__builtin_isfinite(v)) ++bad;
      if (__builtin_isfinite(v)) amax = fmaxf(amax, fabsf(v));
    }
    for (int o = 1; o < 64; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    const float sc = quant_scale(amax);
    for (int j = lane; j < tile; j += 64) {
      const int64_t k = k0 + j;
      const float v = k < in_f ? quant_weight<MODE>(p, row, k, in_f, t, nt, true) : 0.0f;
      if (k < ldc) codes[row * ldc + k] = (uint8_t)quant_encode(v, sc, sb, so);
    }
    if (lane == 0) scales[row * nt + t] = sc;
  }
  quant_count(bad, nonfinite);
}

bool quant_aligned(const void* p, uintptr_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

template <int MODE>
int quant_launch(const QuantSrc& p, int64_t out_f, int64_t in_f, int64_t tile, int64_t ldc, const uint8_t* order,
                 const float* bounds, uint8_t* codes, float* scales, unsigned long long* nonfinite,
                 hipStream_t stream) {
  const int64_t nt = (in_f + tile - 1) / tile;
  hipLaunchKernelGGL(quant_clear_kernel, dim3(1), dim3(1), 0, stream, nonfinite);
  int rc = check_launch("quant_clear_kernel");
  if (rc) return rc;
  const bool pow2 = (tile & (tile - 1)) == 0;
  const bool vec = pow2 && tile >= 4 && tile <= 256 && in_f % 4 == 0 && ldc % 4 == 0 && quant_aligned(codes, 4) &&
                   quant_aligned(p.w, 16) && quant_aligned(p.codes, 4) && quant_aligned(p.update, 16) &&
                   quant_aligned(p.m, 16) && quant_aligned(p.g, p.g_bf16 ? 8 : 16);
  const bool seg = !vec && tile <= 64 && pow2;
  const int64_t per_wave = vec ? 256 / tile : seg ? 64 / tile : 1;
  const int64_t units = out_f * ((nt + per_wave - 1) / per_wave);
  const int64_t blocks = (units * 64 + QUANT_THREADS - 1) / QUANT_THREADS;
  if (blocks > 2147483647LL) return fail(SMAUL_ERR_UNSUPPORTED, "quantize_tiles: matrix too large");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(QUANT_THREADS), 0, stream, p, out_f, in_f, (int)tile, nt,
                       ldc, order, bounds, codes, scales, nonfinite, units);
  };
  if (vec)
    go(quant_vec_kernel<MODE>);
  else if (seg)
    go(quant_tiles_kernel<MODE, true>);
  else
    go(quant_tiles_kernel<MODE, false>);
  return check_launch("quant_tiles_kernel");
}

int quant_check(int64_t out_f, int64_t in_f, int64_t tile, const char* what) {
  if (tile <= 0) return fail(SMAUL_ERR_INVALID, "%s: tile must be > 0, got %lld", what, (long long)tile);
  if (out_f <= 0 || in_f <= 0)
    return fail(SMAUL_ERR_INVALID, "%s: out_f/in_f must be positive, got %lld/%lld", what, (long long)out_f,
                (long long)in_f);
  if (tile > (1 << 20)) return fail(SMAUL_ERR_UNSUPPORTED, "%s: tile too large", what);
  return SMAUL_OK;
}

}  // namespace

extern "C" {

int smaul_fp8_quantize_tiles(const float* w, int64_t out_f, int64_t in_f, int64_t tile, const uint8_t* order,
                             const float* bounds, uint8_t* codes, int64_t ldc, float* scales,
                             unsigned long long* nonfinite, hipStream_t stream) {
  const int rc = quant_check(out_f, in_f, tile, "quantize_tiles");
  if (rc == SMAUL_ERR_INVALID) return rc;
  const int64_t nt = (in_f + tile - 1) / tile;
  if (ldc < nt * tile) return fail(SMAUL_ERR_INVALID, "quantize_tiles: ldc %lld < nt*tile %lld", (long long)ldc,
                                   (long long)(nt * tile));
  if (rc) return rc;
  if (!w || !order || !bounds || !codes || !scales || !nonfinite)
    return fail(SMAUL_ERR_INVALID, "quantize_tiles: null pointer");
  QuantSrc p{};
  p.w = w;
  return quant_launch<QS_MATRIX>(p, out_f, in_f, tile, ldc, order, bounds, codes, scales, nonfinite, stream);
}

int smaul_fp8_requant(const uint8_t* w8, const float* sc, int64_t out_f, int64_t in_f, int64_t tile,
                      const float* update, int decay, float keep, const void* g, int g_dtype, float* m, float lr,
                      float b1, float c1, float b2, float c2, const uint8_t* order, const float* bounds,
                      uint8_t* codes, float* scales, unsigned long long* nonfinite, hipStream_t stream) {
  const int rc = quant_check(out_f, in_f, tile, "requant");
  if (rc) return rc;
  if (!w8 || !sc || !order || !bounds || !codes || !scales || !nonfinite)
    return fail(SMAUL_ERR_INVALID, "requant: null pointer");
  if ((g == nullptr) != (m == nullptr) || (g && update))
    return fail(SMAUL_ERR_INVALID, "requant: g and m go together, and without an update");
  if (g && g_dtype != SMAUL_DTYPE_F32 && g_dtype != SMAUL_DTYPE_BF16)
    return fail(SMAUL_ERR_INVALID, "requant: g must be f32 or bf16");
  QuantSrc p{};
  p.codes = w8;
  p.scales = sc;
  p.update = update;
  p.g = g;
  p.m = m;
  p.g_bf16 = g && g_dtype == SMAUL_DTYPE_BF16;
  p.decay = decay;
  p.keep = keep;
  p.lr = lr;
  p.b1 = b1;
  p.c1 = c1;
  p.b2 = b2;
  p.c2 = c2;
  if (g) return quant_launch<QS_LION>(p, out_f, in_f, tile, in_f, order, bounds, codes, scales, nonfinite, stream);
  return quant_launch<QS_REQUANT>(p, out_f, in_f, tile, in_f, order, bounds, codes, scales, nonfinite, stream);
}

}  // extern "C"
