// backward.hip -- the gradients of the tiled-FP8 linear on MI355X (gfx950).
//
// The input gradient:
//
// dx[r, i] = sum_o g[r, o] * W[o, i] with W[o, i] = lut[w[o, i]] * s[o, i / tile]:
// the backend entry fp8_backward_input (kernel/compute.py:145-153), replacing
// the reference's native kernel kernel/fp8_cpu.cpp:167-259.  Training only;
// not on the forward path.
//
// Two kernels, each a workgroup per 64 x 64 (or 32 x 64) tile of dx walking the
// output dimension o in chunks, whose sums over o run in another order than
// the reference's eight-way split: results agree to fp32 rounding (relative
// 1e-6), not bitwise.
//  - fp8_backward_input_mfma_kernel (tile a multiple of 64, so the tile's 64
//    input columns share one scale column kb): dx[r, i] = sum_o (g[r, o] *
//    s[o, kb]) * lut[w[o, i]].  The products g * s are formed in fp32 and
//    split exactly into three bf16 terms, the codes decode exactly to bf16,
//    so every matrix-core product is exact and the sums are fp32.  (The
//    reference rounds lut * s instead of g * s: the same to fp32 rounding.)
//  - fp8_backward_input_kernel (any tile): the chunk of W decoded to fp32
//    (lut * s rounded once, as the reference's fast path forms it) and of g
//    staged in LDS, each thread a 4 x 4 block of fused multiply-adds.
//
// The weight gradient (fp8_weight_grad_kernel): gw += g^T x, the sums in fp32,
// rounded once into the bf16 accumulator (kernel/fp8_tile.py:172-197).
#include "e4m3.h"
#include "smaul_common.h"

using smaul::check_launch;
using smaul::cu_count;
using smaul::fail;

namespace {

constexpr float e4m3_value(int c) {
  const int e = (c >> 3) & 15, m = c & 7;
  float mag = 0.0f;
  if (e == 15 && m == 7) {
    mag = 448.0f;
  } else if (e == 0) {
    mag = (float)m / 512.0f;
  } else {
    float p = 1.0f;
    for (int i = 7; i < e; ++i) p *= 2.0f;
    for (int i = e; i < 7; ++i) p *= 0.5f;
    mag = (1.0f + (float)m / 8.0f) * p;
  }
  return (c & 128) ? -mag : mag;
}

struct Lut {
  float v[256];
  constexpr Lut() : v() {
    for (int c = 0; c < 256; ++c) v[c] = e4m3_value(c);
  }
};
__constant__ Lut kLut = Lut();

constexpr int BW_T = 64;   // dx tile: rows and input columns
constexpr int BW_K = 32;   // output dimension per LDS chunk

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Four waves, each 32 rows x 32 columns of the tile (v_mfma_f32_32x32x16_bf16:
// lane l holds row / column l % 32 of the operands at k = 8 (l / 32) + 0..7,
// and column l % 32, rows (r / 4) 8 + (l / 32) 4 + r % 4 of the sums).  Per
// chunk of BK o: every thread turns 16 values of g * s (one row, 16
// consecutive o) into their three bf16 terms and writes them to LDS, and
// transposes a 4 x 4 block of codes (4 o x 4 columns, v_perm) into four
// column words of 4 o; the loads of the next chunk are issued before the
// chunk's MFMAs.  VEC: g rows and code rows are
// 16-byte aligned and whole chunks are in range (out_f % 64 == 0, in_f % 64
// == 0), so they load as 16-byte vectors.
//
// BM = 64: the four waves are 2 x 2 over the tile, chunks of 64 o.  BM = 32, for
// grids that leave CUs without a tile: two waves over the columns and two over
// the halves of a chunk of 128 o (their sums meet in LDS), so a tile takes half
// the steps and there are twice as many.
template <bool CANON, bool VEC, int BM>
__global__ void __launch_bounds__(256)
fp8_backward_input_mfma_kernel(const float* __restrict__ g, const uint8_t* __restrict__ w,
                               const float* __restrict__ s, float* __restrict__ dx, int64_t rows, int64_t in_f,
                               int64_t out_f, int64_t tile, int64_t nt) {
  constexpr int BK = 4096 / BM;  // o per chunk
  __shared__ __attribute__((aligned(16))) uint16_t sa[3][BM][BK + 8];  // terms of g * s, [row][o]
  // codes, [column][o]; rows of 72 (136) bytes: the word writes of a wave meet
  // at most two to a bank, the 8-byte fragment reads none
  __shared__ __attribute__((aligned(16))) uint8_t sw[BW_T][BK + 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = BM == 64 ? wave >> 1 : 0, wn = wave & 1, wk = BM == 64 ? 0 : wave >> 1;
  // Workgroup b runs on XCD b % 8: each XCD takes a contiguous band of the
  // tiles in row order, so the column tiles that read the same g rows share
  // one L2 (in launch order they went to eight L2s, with a 38 % hit rate at
  // config 2's gate shape)
  int64_t r0, c0;
  {
    const int64_t nc = gridDim.x, total = nc * gridDim.y, full = (total / 8) * 8;
    int64_t lin = (int64_t)blockIdx.y * nc + blockIdx.x;
    if (lin < full) lin = (lin % 8) * (full / 8) + lin / 8;
    r0 = (lin / nc) * BM;
    c0 = (lin % nc) * BW_T;
  }
  const int64_t kb = c0 / tile;
  // this thread's staging: g row ar, 16 o from ao; codes of o wo..wo+3 x columns wc..wc+3
  constexpr int TPR = BK / 16, NC = BK / 64;  // threads per g row, code blocks per thread
  const int ar = tid / TPR, ao = (tid & (TPR - 1)) * 16;
  const int wo = (tid >> 4) * 4, wc = (tid & 15) * 4;  // code block b: o + 64 b
  const int64_t gr = r0 + ar;
  float gv[16], sv[16];
  uint32_t cw[NC][4];  // row wo + r, columns wc..wc+3 (byte c = column wc + c)
  auto load = [&](int64_t o0) {
    if constexpr (VEC) {
      const float4* gp = (const float4*)(g + (gr < rows ? gr : rows - 1) * out_f + o0 + ao);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 v = gp[q];
        gv[4 * q] = v.x;
        gv[4 * q + 1] = v.y;
        gv[4 * q + 2] = v.z;
        gv[4 * q + 3] = v.w;
      }
      // the wave's lanes hold the chunk's scales, lane l those of o = (l % TPR) * 16 + l / TPR
      // (+ 8), and each lane gathers its 16 (ao = (l % TPR) * 16) with cross-lane reads (written as
      // remainders, not masks, the kernel comes out 6 % slower)
      float sl[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) sl[q] = s[(o0 + (lane & (TPR - 1)) * 16 + lane / TPR + 8 * q) * nt + kb];
#pragma unroll
      for (int j = 0; j < 16; ++j)
        sv[j] = __shfl(sl[NC == 1 ? 0 : j >> 3], (j % (16 / NC)) * TPR | (lane & (TPR - 1)), 64);
#pragma unroll
      for (int b = 0; b < NC; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) cw[b][r] = *(const uint32_t*)(w + (o0 + 64 * b + wo + r) * in_f + c0 + wc);
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int64_t o = o0 + ao + j;
        gv[j] = (gr < rows && o < out_f) ? g[gr * out_f + o] : 0.0f;
        sv[j] = o < out_f ? s[o * nt + kb] : 0.0f;
      }
#pragma unroll
      for (int b = 0; b < NC; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t o = o0 + 64 * b + wo + r;
          uint32_t v = 0;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int64_t i = c0 + wc + c;
            v |= ((o < out_f && i < in_f) ? (uint32_t)w[o * in_f + i] : 0u) << (8 * c);  // code 0 decodes to +0
          }
          cw[b][r] = v;
        }
    }
  };
  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  load(0);
  for (int64_t o0 = 0; o0 < out_f; o0 += BK) {
    {
      uint32_t t[3][8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        float a = gv[2 * q] * sv[2 * q], b = gv[2 * q + 1] * sv[2 * q + 1];
#pragma unroll
        for (int p = 0; p < 3; ++p) {  // term p: the bf16 rounding of what terms < p leave (exact differences)
          t[p][q] = pack_bf16(a, b);
          a = a - bf2f(t[p][q] & 0xffffu);
          b = b - bf2f(t[p][q] >> 16);
        }
      }
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        *(uint4*)&sa[p][ar][ao] = make_uint4(t[p][0], t[p][1], t[p][2], t[p][3]);
        *(uint4*)&sa[p][ar][ao + 8] = make_uint4(t[p][4], t[p][5], t[p][6], t[p][7]);
      }
      // 4 x 4 byte transpose: column word c = (row 0 byte c, ..., row 3 byte c)
      // (v_perm: selector bytes 0-3 pick from the second operand, 4-7 from the first)
#pragma unroll
      for (int b = 0; b < NC; ++b) {
        const uint32_t lo01 = __builtin_amdgcn_perm(cw[b][1], cw[b][0], 0x05010400u);
        const uint32_t hi01 = __builtin_amdgcn_perm(cw[b][1], cw[b][0], 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(cw[b][3], cw[b][2], 0x05010400u);
        const uint32_t hi23 = __builtin_amdgcn_perm(cw[b][3], cw[b][2], 0x07030602u);
        *(uint32_t*)&sw[wc + 0][64 * b + wo] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
        *(uint32_t*)&sw[wc + 1][64 * b + wo] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
        *(uint32_t*)&sw[wc + 2][64 * b + wo] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
        *(uint32_t*)&sw[wc + 3][64 * b + wo] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
      }
    }
    __syncthreads();
    if (o0 + BK < out_f) load(o0 + BK);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int ob = wk * 64 + ks * 16 + (lane >> 5) * 8;
      const int fr = wm * 32 + (lane & 31), fc = wn * 32 + (lane & 31);
      const uint2 c = *(const uint2*)&sw[fc][ob];
      uint32_t d[4];
      decode4<CANON>(c.x, d[0], d[1]);
      decode4<CANON>(c.y, d[2], d[3]);
      const bf16x8_t bf = __builtin_bit_cast(bf16x8_t, make_uint4(d[0], d[1], d[2], d[3]));
#pragma unroll
      for (int p = 0; p < 3; ++p)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8_t*)&sa[p][fr][ob], bf, acc, 0, 0, 0);
    }
    __syncthreads();
  }
  if constexpr (BM == 32) {  // the upper half's sums to the lower half's wave, through sa
    float* part = (float*)&sa[0][0][0];
    static_assert(sizeof(sa) >= 2 * 16 * 64 * 4, "partial sums fit the staging rows");
    if (wk == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) part[(wn * 16 + r) * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (wk == 1) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = acc[r] + part[(wn * 16 + r) * 64 + lane];
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t row = r0 + wm * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
    const int64_t col = c0 + wn * 32 + (lane & 31);
    if (row < rows && col < in_f) dx[row * in_f + col] = acc[r];
  }
}

__global__ void __launch_bounds__(256)
fp8_backward_input_kernel(const float* __restrict__ g, const uint8_t* __restrict__ w, const float* __restrict__ s,
                          float* __restrict__ dx, int64_t rows, int64_t in_f, int64_t out_f, int64_t tile,
                          int64_t nt) {
  __shared__ float sg[BW_K][BW_T + 4];  // g chunk, [o][row]
  __shared__ float sw[BW_K][BW_T + 4];  // decoded W chunk, [o][col]
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int64_t r0 = (int64_t)blockIdx.y * BW_T, c0 = (int64_t)blockIdx.x * BW_T;
  float acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = 0.0f;
  for (int64_t o0 = 0; o0 < out_f; o0 += BW_K) {
    // 32 x 64 of each: 8 loads per thread per operand, coalesced along o for g
    // and along i for w
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int idx = tid + q * 256;
      {
        const int ko = idx & (BW_K - 1), rr = idx >> 5;
        const int64_t r = r0 + rr, o = o0 + ko;
        sg[ko][rr] = (r < rows && o < out_f) ? g[r * out_f + o] : 0.0f;
      }
      {
        const int cc = idx & (BW_T - 1), ko = idx >> 6;
        const int64_t i = c0 + cc, o = o0 + ko;
        float v = 0.0f;
        if (i < in_f && o < out_f) v = kLut.v[w[o * in_f + i]] * s[o * nt + i / tile];
        sw[ko][cc] = v;
      }
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < BW_K; ++k) {
      float gv[4], wv[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) gv[a] = sg[k][ty * 4 + a];
#pragma unroll
      for (int b = 0; b < 4; ++b) wv[b] = sw[k][tx * 4 + b];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_fmaf(gv[a], wv[b], acc[a][b]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int64_t r = r0 + ty * 4 + a;
    if (r >= rows) continue;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int64_t i = c0 + tx * 4 + b;
      if (i < in_f) dx[r * in_f + i] = acc[a][b];
    }
  }
}

// gw[o, i] = bf16(gw[o, i] + sum_r g[r, o] x[r, i]), the sum in fp32 on
// v_mfma_f32_32x32x2_f32.  That instruction wants, per lane, one o (or i) of
// one row, and g and x are row-major: a wave's operand is two rows' 32
// consecutive values as they lie in memory, so both go from global memory to
// registers without LDS.  A workgroup owns 32 NT x 32 NT outputs; each of its
// four waves all of them over every fourth chunk of WG_U row pairs (the next
// chunk's loads in flight), and the four partial sums meet in LDS in wave
// order.
//
// What bounds it: the fp32 matrix rate, 256 FLOP per cycle and CU, on the CUs
// that the 64 x 64 tiles reach (160 at 1280 x 512, so 98 TFLOP/s of the 157).
// 1024 rows, 1280 x 512: one launch of 28 us (46 TFLOP/s; 4096 rows 87 us, 62)
// against 20 library GEMMs of 64 output rows and 20 adds, 424 us; the error
// against float64 is that of the bf16 rounding, 1.66e-3, both ways.
constexpr int WG_U = 8;   // row pairs whose operands are loaded together

template <typename X>
__device__ __forceinline__ float wg_load(const X* p) {
  if constexpr (sizeof(X) == 4)
    return *p;
  else
    return bf2f(*p);
}

template <typename X, int NT>
__global__ void __launch_bounds__(256)
fp8_weight_grad_kernel(const float* __restrict__ g, const X* __restrict__ x, uint16_t* __restrict__ gw, int64_t rows,
                       int64_t out_f, int64_t in_f, int fresh) {
  constexpr int WG_T = 32 * NT;             // outputs of a side
  __shared__ float part[4][16 * NT * NT][64];  // [wave][accumulator][lane]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned nx = (unsigned)((in_f + WG_T - 1) / WG_T);  // the tiles in one dimension, those of a row together
  const int64_t o0 = (int64_t)(blockIdx.x / nx) * WG_T, i0 = (int64_t)(blockIdx.x % nx) * WG_T;
  // outputs past the edge read the last column and are not stored; offsets
  // from the first row of a pair (a lane of the upper half is one row on)
  int64_t oc[NT], ic[NT];
#pragma unroll
  for (int p = 0; p < NT; ++p) {
    const int64_t o = o0 + p * 32 + (lane & 31), i = i0 + p * 32 + (lane & 31);
    oc[p] = (o < out_f ? o : out_f - 1) + (lane >> 5) * out_f;
    ic[p] = (i < in_f ? i : in_f - 1) + (lane >> 5) * in_f;
  }
  f32x16_t acc[NT][NT];
#pragma unroll
  for (int p = 0; p < NT; ++p)
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[p][q][r] = 0.0f;
  float a[2][WG_U][NT], b[2][WG_U][NT];
  const int64_t chunks = (rows + 2 * WG_U - 1) / (2 * WG_U);
  auto load = [&](int set, int64_t c) {
    const int64_t r0 = c * 2 * WG_U;
    const float* gr = g + r0 * out_f;
    const X* xr = x + r0 * in_f;
    if (r0 + 2 * WG_U <= rows) {
#pragma unroll
      for (int u = 0; u < WG_U; ++u, gr += 2 * out_f, xr += 2 * in_f)
#pragma unroll
        for (int p = 0; p < NT; ++p) {
          a[set][u][p] = gr[oc[p]];
          b[set][u][p] = wg_load(xr + ic[p]);
        }
      return;
    }
#pragma unroll
    for (int u = 0; u < WG_U; ++u, gr += 2 * out_f, xr += 2 * in_f) {
      const bool in = r0 + 2 * u + (lane >> 5) < rows;
#pragma unroll
      for (int p = 0; p < NT; ++p) {
        a[set][u][p] = in ? gr[oc[p]] : 0.0f;
        b[set][u][p] = in ? wg_load(xr + ic[p]) : 0.0f;
      }
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int u = 0; u < WG_U; ++u)
#pragma unroll
      for (int p = 0; p < NT; ++p)
#pragma unroll
        for (int q = 0; q < NT; ++q)
          acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[set][u][p], b[set][u][q], acc[p][q], 0, 0, 0);
  };
  int64_t c = wave;
  if (c < chunks) load(0, c);
  for (; c < chunks; c += 8) {  // chunks past the end load zeros
    load(1, c + 4);
    multiply(0);
    load(0, c + 8);
    multiply(1);
  }
#pragma unroll
  for (int p = 0; p < NT; ++p)
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[wave][(p * NT + q) * 16 + r][lane] = acc[p][q][r];
  __syncthreads();
  // each wave finishes a quarter of the accumulators
#pragma unroll
  for (int r4 = 0; r4 < 4 * NT * NT; ++r4) {
    const int n = wave * 4 * NT * NT + r4, p = n / (16 * NT), q = n / 16 % NT, r = n % 16;
    const float sum = part[0][n][lane] + part[1][n][lane] + part[2][n][lane] + part[3][n][lane];
    const int64_t o = o0 + p * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3), i = i0 + q * 32 + (lane & 31);
    if (o < out_f && i < in_f) {
      uint16_t* d = gw + o * in_f + i;
      *d = (uint16_t)pack_bf16((fresh ? 0.0f : bf2f(*d)) + sum, 0.0f);
    }
  }
}

// ---- SwiGLU product of the training path (model.py:289-290) -----------------
// out = silu(g) * u and its gradients, fp32 arithmetic whatever the dtype, each
// one pass where the tensor operations take two and four (with the fp32
// intermediates between them), every rounding where theirs is.  HBM-bound: 3 and
// 5 tensors' bytes.
template <typename X>
__device__ __forceinline__ void sg_store(X* p, float v) {
  if constexpr (sizeof(X) == 4)
    *p = v;
  else
    *p = (uint16_t)pack_bf16(v, 0.0f);
}

template <typename X, bool BACK>
__global__ void __launch_bounds__(256)
swiglu_kernel(const X* __restrict__ g, const X* __restrict__ u, const X* __restrict__ dout, X* __restrict__ a,
              X* __restrict__ b, int64_t n) {
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x); i < n; i += (int64_t)gridDim.x * 256) {
    const float gv = wg_load(g + i), uv = wg_load(u + i);
    const float e = 1.0f + expf(-gv), silu = gv / e;  // one rounding, where g * (1 / e) has two
    if constexpr (BACK) {
      const float d = wg_load(dout + i), sig = 1.0f / e;
      sg_store(a + i, d * uv * sig * __builtin_fmaf(gv, 1.0f - sig, 1.0f));
      sg_store(b + i, d * silu);
    } else {
      sg_store(a + i, silu * uv);
    }
  }
}

template <bool BACK>
int swiglu_launch(const void* g, const void* u, const void* dout, void* a, void* b, int64_t n, int dtype,
                  hipStream_t stream) {
  const unsigned blocks = (unsigned)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  if (dtype == SMAUL_DTYPE_F32)
    hipLaunchKernelGGL((swiglu_kernel<float, BACK>), dim3(blocks), dim3(256), 0, stream, (const float*)g,
                       (const float*)u, (const float*)dout, (float*)a, (float*)b, n);
  else
    hipLaunchKernelGGL((swiglu_kernel<uint16_t, BACK>), dim3(blocks), dim3(256), 0, stream, (const uint16_t*)g,
                       (const uint16_t*)u, (const uint16_t*)dout, (uint16_t*)a, (uint16_t*)b, n);
  return check_launch("swiglu_kernel");
}

}  // namespace

extern "C" {

int smaul_fp8_backward_input(const float* g, const uint8_t* w, const float* s, float* dx, int64_t rows,
                             int64_t in_f, int64_t out_f, int64_t tile, hipStream_t stream) {
  // in_f / out_f may be 0, as in the reference (fp8_cpu.cpp:227-228): no
  // columns, or an empty sum (dx all zeros, g / w / s not read)
  if (tile <= 0 || in_f < 0 || out_f < 0 || rows < 0)
    return fail(SMAUL_ERR_INVALID, "fp8_backward_input: need tile > 0 and in_f, out_f, rows >= 0, got %lld/%lld/%lld",
                (long long)tile, (long long)in_f, (long long)out_f);
  if (rows == 0 || in_f == 0) return SMAUL_OK;
  if (!dx || (out_f > 0 && (!g || !w || !s))) return fail(SMAUL_ERR_INVALID, "fp8_backward_input: null pointer");
  const int64_t gx = (in_f + BW_T - 1) / BW_T, gy = (rows + BW_T - 1) / BW_T;
  if (gx > 2147483647LL || gy > 65535) return fail(SMAUL_ERR_UNSUPPORTED, "fp8_backward_input: grid too large");
  const int64_t nt = (in_f + tile - 1) / tile;
  if (tile % BW_T == 0) {  // a dx tile's columns share one scale column
    // VEC reads its first chunk unguarded, so an empty sum goes to the guarded kernel
    const bool vec = out_f > 0 && out_f % 64 == 0 && in_f % BW_T == 0 && ((uintptr_t)g & 15) == 0 &&
                     ((uintptr_t)w & 15) == 0;
    // BM = 32 under two 64-row tiles a CU, or half a one for the guarded loads,
    // which twice the tiles repeat and which want more than one chunk to fill
    // (64 / 32 rows, us, tiles of 64 rows in brackets): vector 1000 x 1280 -> 512
    // (128) 26.3 / 17.0, 3000 (376) 35.2 / 28.5, 1000 x 5120 -> 2048 (512) 134 / 142,
    // 3000 x 512 -> 1280 (940) 25.6 / 28.5; guarded 500 x 777 -> 1000 (128) 48.0
    // / 36.6, 1000 (256) 48.1 / 48.5, 3000 x 300 -> 200 (188) 19.9 / 22.2,
    // 20000 x 10000 -> 192 (939) 1703 / 2361, 64 x 32 -> 512 (8) 6.4 / 6.6
    const int64_t tiles = gx * gy, cus = cu_count();
    const bool small = vec ? out_f % 128 == 0 && tiles < 2 * cus : out_f > 64 && 2 * tiles <= cus;
    auto go = [&](auto kernel, int64_t grid_y) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)gx, (unsigned)grid_y), dim3(256), 0, stream, g, w, s, dx, rows, in_f,
                         out_f, tile, nt);
    };
    if (small)
      vec ? go(fp8_backward_input_mfma_kernel<false, true, 32>, (rows + 31) / 32)
          : go(fp8_backward_input_mfma_kernel<false, false, 32>, (rows + 31) / 32);
    else
      vec ? go(fp8_backward_input_mfma_kernel<false, true, 64>, gy)
          : go(fp8_backward_input_mfma_kernel<false, false, 64>, gy);
    return check_launch("fp8_backward_input_mfma_kernel");
  }
  hipLaunchKernelGGL(fp8_backward_input_kernel, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, stream, g, w, s, dx,
                     rows, in_f, out_f, tile, nt);
  return check_launch("fp8_backward_input_kernel");
}

int smaul_fp8_weight_grad(const float* g, const void* x, int x_dtype, void* gw, int64_t rows, int64_t in_f,
                          int64_t out_f, int fresh, hipStream_t stream) {
  if (in_f < 0 || out_f < 0 || rows < 0)
    return fail(SMAUL_ERR_INVALID, "fp8_weight_grad: need in_f, out_f, rows >= 0, got %lld/%lld/%lld",
                (long long)in_f, (long long)out_f, (long long)rows);
  if (x_dtype != SMAUL_DTYPE_F32 && x_dtype != SMAUL_DTYPE_BF16)
    return fail(SMAUL_ERR_INVALID, "fp8_weight_grad: x must be f32 or bf16");
  if (in_f == 0 || out_f == 0 || (rows == 0 && !fresh)) return SMAUL_OK;
  if (!gw || (rows > 0 && (!g || !x))) return fail(SMAUL_ERR_INVALID, "fp8_weight_grad: null pointer");
  const int64_t tiles = ((in_f + 63) / 64) * ((out_f + 63) / 64);
  // 32 x 32 outputs where 64 x 64 leave half of the CUs idle (64 / 32, us: 64
  // rows, 640 x 256 8.8 / 5.3, 1024 rows 25.0 / 10.4, 3000 rows 65.5 / 26.5; 160
  // tiles: 1024 rows, 1280 x 512 28.6 / 29.8, 4096 rows 86 / 98)
  const int64_t side = 2 * tiles < cu_count() ? 32 : 64;
  const int64_t blocks = ((in_f + side - 1) / side) * ((out_f + side - 1) / side);
  // a launch dimension holds fewer than 2^32 threads: 6e10 weights, of any shape
  if (blocks >= (1LL << 32) / 256) return fail(SMAUL_ERR_UNSUPPORTED, "fp8_weight_grad: matrix too large");
  const dim3 grid((unsigned)blocks);
  auto go = [&](auto kernel, auto* xp) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, g, xp, (uint16_t*)gw, rows, out_f, in_f, fresh);
  };
  if (x_dtype == SMAUL_DTYPE_F32)
    side == 32 ? go(fp8_weight_grad_kernel<float, 1>, (const float*)x)
               : go(fp8_weight_grad_kernel<float, 2>, (const float*)x);
  else
    side == 32 ? go(fp8_weight_grad_kernel<uint16_t, 1>, (const uint16_t*)x)
               : go(fp8_weight_grad_kernel<uint16_t, 2>, (const uint16_t*)x);
  return check_launch("fp8_weight_grad_kernel");
}

int smaul_swiglu(const void* g, const void* u, void* out, int64_t n, int dtype, hipStream_t stream) {
  if (n < 0 || (dtype != SMAUL_DTYPE_F32 && dtype != SMAUL_DTYPE_BF16))
    return fail(SMAUL_ERR_INVALID, "swiglu: need n >= 0 and f32|bf16");
  if (n == 0) return SMAUL_OK;
  if (!g || !u || !out) return fail(SMAUL_ERR_INVALID, "swiglu: null pointer");
  return swiglu_launch<false>(g, u, nullptr, out, nullptr, n, dtype, stream);
}

int smaul_swiglu_backward(const void* dout, const void* g, const void* u, void* dg, void* du, int64_t n, int dtype,
                          hipStream_t stream) {
  if (n < 0 || (dtype != SMAUL_DTYPE_F32 && dtype != SMAUL_DTYPE_BF16))
    return fail(SMAUL_ERR_INVALID, "swiglu_backward: need n >= 0 and f32|bf16");
  if (n == 0) return SMAUL_OK;
  if (!dout || !g || !u || !dg || !du) return fail(SMAUL_ERR_INVALID, "swiglu_backward: null pointer");
  return swiglu_launch<true>(g, u, dout, dg, du, n, dtype, stream);
}

}  // extern "C"
