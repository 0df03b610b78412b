// attn.hip -- the linear-attention recurrence of SmaulLinear on MI355X (gfx950).
//
// Replaces the reference's native CPU kernels kernel/attn_cpu.cpp
// (attn_forward :144-212, attn_step :421-492, attn_backward :227-368) behind
// the backend entries attn_forward / attn_step / attn_backward
// (kernel/compute.py:265-322).  Per (batch, head):
//   kn_t = k_t / max(||k_t||, 1e-6)          ||k_t|| accumulated in double
//   S_t = S_{t-1} + kn_t (x) v_t,  z_t = z_{t-1} + kn_t
//   num_t = q_t @ S_t,  den_t = max(q_t . z_t, eps),  y_t = num_t / den_t
// Layouts: Q/K/V/Y [B,T,H,D] fp32, DEN [B,T,H], S [B,H,D,D] (row i is the key
// index), z [B,H,D].
//
// The results are bit-identical to the reference kernel: every (b, h) runs
// its T steps in order, each sum runs sequentially over i with a separate
// multiply and add (the library is built with -ffp-contract=off), the key
// norm is a sequential double sum, and the division and square root are
// correctly rounded.  Element (i, j) of S and entry j of num are owned by one
// thread (column j), so the reference's per-element order holds exactly.
//
// For D <= 128 (every preset of the reference: model.py:1020-1085) the forward
// and the backward run as systolic arrays over (row, step) that keep every
// sum's order (below), the forward of many short tasks with a workgroup per
// (b, h) task and S in registers (attn_use_array); larger D (the reference
// accepts D <= 2048) keeps S in global memory, the caller's S_out or a
// workspace, with one workgroup per task.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "smaul_common.h"

using smaul::check_launch;
using smaul::cu_count;
using smaul::fail;

namespace {

// 1 / max(||k||, 1e-6) of one key (attn_cpu.cpp:40-51): the norm summed in
// double in index order, rounded to fp32, clamped, one fp32 reciprocal.
__device__ __forceinline__ float attn_inv_norm2(double n2) {
  const float n = (float)__builtin_sqrt(n2);
  const float nc = (!__builtin_isfinite(n) || n < 1e-6f) ? 1e-6f : n;
  return 1.0f / nc;
}

// n2 plus the squares of k[i .. end), in order, read 16 ahead of the sum
__device__ __forceinline__ double attn_square_sum(double n2, const float* k, int i, int end) {
  for (; i + 16 <= end; i += 16) {
    float kk[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) kk[u] = k[i + u];
#pragma unroll
    for (int u = 0; u < 16; ++u) n2 = n2 + (double)kk[u] * (double)kk[u];
  }
  for (; i < end; ++i) {
    const double ki = (double)k[i];
    n2 = n2 + ki * ki;
  }
  return n2;
}

__device__ __forceinline__ float attn_inv_norm(const float* k, int D) {
  return attn_inv_norm2(attn_square_sum(0.0, k, 0, D));
}

// ---------------------------------------------------------------------------
// D <= 128: a systolic array over (row i, time t)
// ---------------------------------------------------------------------------
// Step t of row i needs S[i] of step t - 1 and the partial num of row i - 1 at
// step t, and nothing else: along an anti-diagonal of (t, i) every row can
// work at once without touching the reference's order.  Lane i of a wave owns
// row i (RPL consecutive rows for D > 64) of J columns of S in registers and
// at tick tau works on step t = tau - i; num and den move to lane i + 1
// between ticks as the DPP operand of the add itself (wave_shr:1, lane 0
// starts from +0), and leave the array at the lane of row D - 1.  A tick is 4
// VALU operations per column and row (multiply and add kept apart) plus about
// a dozen shared by the columns, and a task of D x D takes T + D ticks on D /
// J waves instead of T * D dependent steps on one.
//
// A workgroup is AC_W such waves on neighbouring columns of one task, one
// wave that stages the next AttnCol::CH steps of q, kn and v meanwhile, and
// one that computes the key norms of the steps after those (a serial double
// sum, one lane per step).  The steps sit in a
// ring, which holds the 64 a wave's lanes are spread over and the
// chunk being written; steps outside [0, T) are zeros, which leave S and z as
// they are (+0 + +-0 = +0, x + +-0 = x).  Row strides (in the units the lanes
// read, 8 or 16 bytes) are chosen odd against the lanes' one-row skew, so the
// reads meet no bank twice.
//
// What bounds it: the length of the array in ticks, T + D, at the issue rate
// of one wave per SIMD (4.6 cycles an instruction, 8.7 an add with a DPP
// operand: about 140 cycles a tick at J = 2).  B 2, T 256, H 8, D 64: 32 us,
// against 990 us with one workgroup per task and one thread per column (16
// workgroups, every thread walking all D rows of a step with three LDS reads
// each); 44 us before the staging was spread over two waves and the operands
// were read a batch ahead.
constexpr int AC_W = 4;                     // computing waves of a workgroup
constexpr int AC_NT = (AC_W + 2) * 64;      // and the staging and the norm wave

// lane i takes lane i - 1's value, lane 0 takes +0
__device__ __forceinline__ float wave_shr1(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}

// LDS written by other lanes of this wave: the hardware runs a wave's LDS
// operations in order, so only the compiler must keep them so
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int N>
using Set = std::integral_constant<int, N>;  // a register set by number, known when compiled

template <int RPL, int J>
struct AttnCol {
  static constexpr int CH = RPL == 1 ? 32 : 16;    // steps staged at once
  static constexpr int RN = RPL == 1 ? 128 : 96;   // steps in the ring, at least 64 + 2 CH
  static constexpr int NB = J == 8 ? 4 : 8;        // ticks whose operands are read together
  static constexpr int CW = AC_W * J;              // columns of a workgroup
  static constexpr int RS = RPL == 1 ? 66 : 132;   // (x, u) pairs of a ring row
  static constexpr int VS = CW + (J == 2 ? 2 : 4); // floats of a ring row of v
  static constexpr int VN = CH * CW / 64;          // v values a staging lane loads per chunk
  __attribute__((aligned(16))) float2 xu[RN * RS];
  __attribute__((aligned(16))) float v[RN * VS];
  float out[AC_W][CH][J + 1];                      // num (J) and den of the chunk's ticks
  float k[2 * CH][64 * RPL + 1];                   // raw keys of the norm wave's two chunks
  float inv[4][CH];                                // 1 / norm of a chunk's keys, by chunk mod 4
};

// REV is the adjoint's column pass of the backward: time runs backwards, the
// state is Dm += q (x) dnum with dnum = V (1 / DEN_in) (V is dY), and what
// leaves the array is dv = Dm^T kn, stored as it is.
template <int RPL, int J, bool REV>
__device__ __forceinline__ void
attn_col(AttnCol<RPL, J>& sm, const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
         const float* __restrict__ DEN_in, float* __restrict__ Y, float* __restrict__ DEN, float* __restrict__ S_out,
         float* __restrict__ z_out, int64_t T, int H, int D, int groups, float eps) {
  using L = AttnCol<RPL, J>;
  constexpr int CH = L::CH, RS = L::RS, VS = L::VS, CW = L::CW, RN = L::RN, NB = L::NB;
  const int64_t task = blockIdx.x / groups;
  const int cg = (int)(blockIdx.x - task * groups);
  const int64_t b = task / H, h = task % H;
  const int tid = threadIdx.x, lane = tid & 63;
  // uniform, so that the two roles are scalar branches and each wave meets its own barriers only
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // stride between steps and the first one
  const int64_t rs = REV ? -(int64_t)H * D : (int64_t)H * D;
  const int64_t base = ((b * T + (REV ? T - 1 : 0)) * H + h) * D;
  const int last = (D - 1) / RPL;             // the lane that holds row D - 1
  const bool half = RPL == 2 && (D & 1);      // whose second row does not exist
  const int64_t chunks = T > 0 ? (T + last + CH - 1) / CH : 0;

  for (int e = tid; e < RN * RS; e += AC_NT) sm.xu[e] = make_float2(0.0f, 0.0f);
  for (int e = tid; e < RN * VS; e += AC_NT) sm.v[e] = 0.0f;

  if (wave == AC_W) {
    // staging wave: lane = column (columns lane, lane + 64) of q and k, the
    // last one again past D (such lanes' values reach no result); steps past
    // T are zero.  Two register sets: the loads of a chunk are issued two
    // periods before its values are written to the ring
    float sq[2][CH * RPL], sk[2][CH * RPL], sv[2][L::VN], sd[2][REV ? L::VN : 1];
    constexpr int VR = 64 / CW;  // rows of v that a load of the wave covers
    const int vr0 = lane / CW;
    uint32_t col[RPL];
#pragma unroll
    for (int p = 0; p < RPL; ++p) col[p] = lane + 64 * p < D ? lane + 64 * p : D - 1;
    const int64_t voff = vr0 * rs + (cg * CW + lane % CW < D ? cg * CW + lane % CW : D - 1);
    const int64_t doff = REV ? (b * T + T - 1 - vr0) * H + h : 0;  // DEN of step vr0
    auto load = [&](auto set, int64_t c) {
      const int64_t left = T - c * CH;  // steps of this chunk on
      if (left >= CH) {
        const float *qr = Q + base + c * CH * rs, *kr = K + base + c * CH * rs;
        const float* vr = V + base + c * CH * rs;
        const float* dr = REV ? DEN_in - c * CH * H : nullptr;
#pragma unroll
        for (int r = 0; r < CH; ++r, qr += rs, kr += rs)
#pragma unroll
          for (int p = 0; p < RPL; ++p) {
            sq[set][r * RPL + p] = qr[col[p]];
            sk[set][r * RPL + p] = kr[col[p]];
          }
#pragma unroll
        for (int n = 0; n < L::VN; ++n, vr += VR * rs) {
          sv[set][n] = vr[voff];
          if constexpr (REV) {
            sd[set][n] = dr[doff];
            dr -= (int64_t)VR * H;
          }
        }
        return;
      }
#pragma unroll
      for (int r = 0; r < CH; ++r) {
        const int64_t o = base + (c * CH + r) * rs;
#pragma unroll
        for (int p = 0; p < RPL; ++p) {
          sq[set][r * RPL + p] = r < left ? Q[o + col[p]] : 0.0f;
          sk[set][r * RPL + p] = r < left ? K[o + col[p]] : 0.0f;
        }
      }
#pragma unroll
      for (int n = 0; n < L::VN; ++n) {
        const int64_t t = c * CH + n * VR;
        const bool in = n * VR + vr0 < left;
        sv[set][n] = in ? V[base + t * rs + voff] : 0.0f;
        if constexpr (REV) sd[set][n] = in ? DEN_in[doff - t * H] : 1.0f;
      }
    };
    auto stage = [&](auto set, int64_t c) {
      const int row0 = (int)(c % (RN / CH)) * CH;
      const float inv = lane < CH ? sm.inv[c & 3][lane] : 0.0f;
#pragma unroll
      for (int r = 0; r < CH; ++r) {
        const float ir = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), r));
#pragma unroll
        for (int p = 0; p < RPL; ++p) {
          const float q = sq[set][r * RPL + p], kn = sk[set][r * RPL + p] * ir;
          sm.xu[(row0 + r) * RS + lane + 64 * p] = REV ? make_float2(kn, q) : make_float2(q, kn);
        }
      }
#pragma unroll
      for (int n = 0; n < L::VN; ++n) {
        sm.v[(row0 + n * VR + vr0) * VS + lane % CW] = REV ? sv[set][n] * (1.0f / sd[set][n]) : sv[set][n];
      }
    };
    if (T > 0) {
      load(Set<0>(), 0);
      load(Set<1>(), 1);
    }
    __syncthreads();
    if (T > 0) {
      stage(Set<0>(), 0);
      load(Set<0>(), 2);
    }
    __syncthreads();
    for (int64_t c = 0; c < chunks; c += 2) {  // period c stages chunk c + 1
      if (c + 1 < chunks) {
        stage(Set<1>(), c + 1);
        load(Set<1>(), c + 3);
      }
      __syncthreads();
      if (c + 1 < chunks) {
        if (c + 2 < chunks) {
          stage(Set<0>(), c + 2);
          load(Set<0>(), c + 4);
        }
        __syncthreads();
      }
    }
    return;
  }

  if (wave == AC_W + 1) {
    // norm wave, lane = step: the norms of chunks 2 m and 2 m + 1 in the two
    // periods that end before period 2 m - 1, which stages the first of them
    float sk[2 * CH * RPL];
    double n2 = 0.0;
    auto load = [&](int64_t m) {
      const int64_t left = T - 2 * m * CH;
      const float* kr = K + base + (left > 0 ? 2 * m * CH : T - 1) * rs;
#pragma unroll
      for (int r = 0; r < 2 * CH; ++r) {
#pragma unroll
        for (int p = 0; p < RPL; ++p) sk[r * RPL + p] = kr[lane + 64 * p < D ? lane + 64 * p : D - 1];
        kr += r + 1 < left ? rs : 0;  // steps past T: the last one again
      }
    };
    const int mid = D / 32 * 16;
    const float* row = sm.k[lane & (2 * CH - 1)];
    auto first_half = [&](int64_t m) {
#pragma unroll
      for (int r = 0; r < 2 * CH; ++r)
#pragma unroll
        for (int p = 0; p < RPL; ++p) sm.k[r][lane + 64 * p] = sk[r * RPL + p];
      wave_lds_fence();
      load(m + 1);
      n2 = attn_square_sum(0.0, row, 0, mid);
    };
    auto second_half = [&](int64_t m) {
      if (lane < 2 * CH) sm.inv[(2 * m + lane / CH) & 3][lane % CH] = attn_inv_norm2(attn_square_sum(n2, row, mid, D));
      wave_lds_fence();
    };
    if (T > 0) {
      load(0);
      first_half(0);
      second_half(0);
    }
    __syncthreads();
    for (int64_t c = -1; c < chunks; ++c) {
      const int64_t m = (c + 3) >> 1;
      if (2 * m < chunks) {
        if (c & 1)
          first_half(m);
        else
          second_half(m);
      }
      __syncthreads();
    }
    return;
  }

  // computing waves: rows lane * RPL .., columns c0 ..
  const int c0 = cg * CW + wave * J;
  float S[RPL][J], z[RPL], num[J], den = 0.0f;
#pragma unroll
  for (int p = 0; p < RPL; ++p) {
    z[p] = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) S[p][j] = 0.0f;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) num[j] = 0.0f;
  __syncthreads();
  __syncthreads();
  for (int64_t c = 0; c < chunks; ++c) {
    // in batches of NB ticks, the operands of the next batch read meanwhile
    const int tick0 = (int)(c % (RN / CH)) * CH;
    float* out = &sm.out[wave][0][0];
    float x[2][NB][RPL], u[2][NB][RPL], v[2][NB][J];
    auto fetch = [&](int set, int tt, int tick) {
      int row = tick0 + tick - lane;
      if constexpr (RN == 128)
        row &= RN - 1;
      else
        row = (int)min((unsigned)row, (unsigned)(row + RN));
      const float* a = (const float*)&sm.xu[row * RS + RPL * lane];
      if constexpr (RPL == 1) {
        const float2 w = *(const float2*)a;
        x[set][tt][0] = w.x;
        u[set][tt][0] = w.y;
      } else {
        const float4 w = *(const float4*)a;
        x[set][tt][0] = w.x;
        u[set][tt][0] = w.y;
        x[set][tt][1] = w.z;
        u[set][tt][1] = w.w;
      }
      if constexpr (J == 2) {
        const float2 w = *(const float2*)&sm.v[row * VS + wave * J];
        v[set][tt][0] = w.x;
        v[set][tt][1] = w.y;
      } else {
#pragma unroll
        for (int j = 0; j < J; j += 4) {
          const float4 w = *(const float4*)&sm.v[row * VS + wave * J + j];
          v[set][tt][j] = w.x;
          v[set][tt][j + 1] = w.y;
          v[set][tt][j + 2] = w.z;
          v[set][tt][j + 3] = w.w;
        }
      }
    };
#pragma unroll
    for (int tt = 0; tt < NB; ++tt) fetch(0, tt, tt);
#pragma unroll
    for (int tt0 = 0; tt0 < CH; tt0 += NB) {
      const int s = (tt0 / NB) & 1;
      float left[NB][J + 1];  // what leaves the array at the lane of row D - 1
#pragma unroll
      for (int tt = 0; tt < NB; ++tt) {
        if (tt0 + NB < CH) fetch(s ^ 1, tt, tt0 + NB + tt);
        // groups of operations that do not depend on one another: a DPP read
        // wants two instructions between it and what it reads
        float g[J], gz = 0.0f;
#pragma unroll
        for (int p = 0; p < RPL; ++p) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < J; ++j) g[j] = u[s][tt][p] * v[s][tt][j];
          if constexpr (!REV) z[p] = z[p] + u[s][tt][p];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < J; ++j) S[p][j] = S[p][j] + g[j];
          if constexpr (!REV) gz = x[s][tt][p] * z[p];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < J; ++j) g[j] = x[s][tt][p] * S[p][j];
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (!REV) {
            den = (p ? den : wave_shr1(den)) + gz;
            left[tt][J] = p && half ? left[tt][J] : den;
          }
#pragma unroll
          for (int j = 0; j < J; ++j) num[j] = (p ? num[j] : wave_shr1(num[j])) + g[j];
#pragma unroll
          for (int j = 0; j < J; ++j) left[tt][j] = p && half ? left[tt][j] : num[j];
        }
      }
      if (lane == last) {
#pragma unroll
        for (int tt = 0; tt < NB; ++tt)
#pragma unroll
          for (int j = 0; j < J + !REV; ++j) out[(tt0 + tt) * (J + 1) + j] = left[tt][j];
      }
    }
    wave_lds_fence();
    const int64_t t = c * CH + lane - last;  // the step that left the array at tick c * CH + lane
    if (lane < CH && t >= 0 && t < T) {
      float denc = 1.0f;
      if constexpr (!REV) {
        const float d = out[lane * (J + 1) + J];
        denc = d < eps ? eps : d;
        if (DEN && c0 == 0) DEN[(b * T + t) * H + h] = denc;
      }
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (c0 + j < D) {
          const float n = out[lane * (J + 1) + j];
          Y[base + t * rs + c0 + j] = REV ? n : n / denc;
        }
    }
    wave_lds_fence();
    __syncthreads();
  }
  if (S_out) {
#pragma unroll
    for (int p = 0; p < RPL; ++p) {
      const int i = lane * RPL + p;
      if (i >= D) continue;
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (c0 + j < D) S_out[(task * D + i) * D + c0 + j] = S[p][j];
      if (c0 == 0) z_out[task * D + i] = z[p];
    }
  }
}

template <int RPL, int J>
__global__ void __launch_bounds__(AC_NT)
attn_fwd_col_kernel(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
                    float* __restrict__ Y, float* __restrict__ DEN, float* __restrict__ S_out,
                    float* __restrict__ z_out, int64_t T, int H, int D, int groups, float eps) {
  __shared__ AttnCol<RPL, J> sm;
  attn_col<RPL, J, false>(sm, Q, K, V, nullptr, Y, DEN, S_out, z_out, T, H, D, groups, eps);
}

// Columns per wave: the fewest of 2, 4, 8 whose workgroups (tasks of them,
// times the passes of one launch) still find a CU each.  A tick costs about
// 4 J + 15 instructions, so fewer columns finish sooner as long as no CU has
// to run two workgroups, and beyond that more of them share the 15.
int attn_col_width(int64_t tasks, int64_t D) {
  for (int j = 2; j < 8; j *= 2)
    if (tasks * ((D + AC_W * j - 1) / (AC_W * j)) <= cu_count()) return j;
  return 8;
}

// ---- D <= 128, many short tasks: a workgroup per task, a thread per column ---
// Thread j owns column j (S[0..D-1][j]) and z[j] in registers; a chunk of
// ATTN_CH steps of q/k/v is staged through LDS, its key norms computed by a
// thread each.  A task is T * D dependent operations, but with 12 KB of LDS (25
// for D > 64) and a wave or two a CU runs many of them at once.
constexpr int ATTN_CH = 16;

template <int DMAX>
__global__ void __launch_bounds__(DMAX)
attn_fwd_reg_kernel(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
                    float* __restrict__ Y, float* __restrict__ DEN, float* __restrict__ S_out,
                    float* __restrict__ z_out, int64_t T, int H, int D, float eps) {
  __shared__ __attribute__((aligned(16))) float s_q[ATTN_CH][DMAX];
  __shared__ __attribute__((aligned(16))) float s_k[ATTN_CH][DMAX];
  __shared__ __attribute__((aligned(16))) float s_v[ATTN_CH][DMAX];
  __shared__ __attribute__((aligned(16))) float s_kn[DMAX];
  __shared__ __attribute__((aligned(16))) float s_z[DMAX];
  __shared__ float s_inv[ATTN_CH];
  const int64_t task = blockIdx.x;
  const int64_t b = task / H, h = task % H;
  const int j = threadIdx.x;
  const bool col = j < D;
  float S[DMAX];
#pragma unroll
  for (int i = 0; i < DMAX; ++i) S[i] = 0.0f;
  float zj = 0.0f;
  const int64_t rs = (int64_t)H * D;          // stride between time steps
  const int64_t base = (b * T * H + h) * D;   // (b, t = 0, h)
  for (int64_t t0 = 0; t0 < T; t0 += ATTN_CH) {
    const int nt = (int)(T - t0 < ATTN_CH ? T - t0 : ATTN_CH);
    // stage the chunk: every thread loads its column of each step
    if (col) {
#pragma unroll
      for (int tt = 0; tt < ATTN_CH; ++tt)
        if (tt < nt) {
          const int64_t o = base + (t0 + tt) * rs + j;
          s_q[tt][j] = Q[o];
          s_k[tt][j] = K[o];
          s_v[tt][j] = V[o];
        }
    }
    __syncthreads();
    if (j < nt) s_inv[j] = attn_inv_norm(s_k[j], D);
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      float vj = 0.0f;
      if (col) {
        const float knj = s_k[tt][j] * s_inv[tt];
        zj = zj + knj;
        s_kn[j] = knj;
        s_z[j] = zj;
        vj = s_v[tt][j];
      }
      __syncthreads();
      float num = 0.0f, den = 0.0f;
#pragma unroll
      for (int i = 0; i < DMAX; ++i) {
        if (i < D) {
          const float qi = s_q[tt][i];
          S[i] = S[i] + s_kn[i] * vj;
          num = num + qi * S[i];
          den = den + qi * s_z[i];
        }
      }
      const float denc = den < eps ? eps : den;
      const int64_t t = t0 + tt;
      if (col) Y[base + t * rs + j] = num / denc;
      if (DEN && j == 0) DEN[(b * T + t) * H + h] = denc;
      __syncthreads();  // s_kn / s_z are rewritten by the next step
    }
  }
  if (col) {
    if (S_out) {
      float* so = S_out + task * D * D + j;
#pragma unroll
      for (int i = 0; i < DMAX; ++i)
        if (i < D) so[(int64_t)i * D] = S[i];
    }
    if (z_out) z_out[task * D + j] = zj;
  }
}

// What `workgroups` of the array measure, in ns: each has a CU to itself (90 to
// 135 KB of LDS) and takes 7500 (clearing the ring, the first loads and norms,
// the drain) and its ticks, whole chunks of them.
double attn_array_ns(int64_t workgroups, int64_t T, int64_t D, int j) {
  const int rpl = D <= 64 ? 1 : 2, ch = rpl == 1 ? AttnCol<1, 2>::CH : AttnCol<2, 2>::CH;
  const double tick = rpl == 1 ? (j == 2 ? 73 : j == 4 ? 94 : 156) : (j == 2 ? 116 : j == 4 ? 160 : 256);
  const int64_t cus = cu_count();
  return (double)((workgroups + cus - 1) / cus) * (7500 + (T + (D - 1) / rpl + ch - 1) / ch * ch * tick);
}

constexpr int64_t ATTN_GRID_THREADS = 1LL << 32;  // a launch dimension holds fewer

// Whether a forward runs as the array: the sooner end of the two from what they
// measure.  A step of the other kernel takes 1200 + 45 D ns while the CUs hide
// one task's latency behind others', beyond that a time per task.  us, array / registers:
//   D 64    T 1: 512 tasks 70 / 12, 16384 2189 / 43    T 4: 8 tasks 15 / 19, 128 25 / 19
//   D 64   T 16: 128 tasks 24 / 64, 512 93 / 68, 16384 2919 / 431
//   D 64  T 256: 8 tasks 31 / 990, 2048 928 / 1154, 16384 7382 / 6907
//   D 128  T 64: 8 tasks 23 / 456, 512 316 / 502, 16384 10000 / 7915
//   D 16   T 64: 8 tasks 15 / 117, 512 47 / 121, 2048 182 / 141, 16384 1440 / 826
bool attn_use_array(int64_t tasks, int64_t T, int64_t D, int j, int64_t groups) {
  if (tasks * groups >= ATTN_GRID_THREADS / AC_NT) return false;
  const double per_task = (D <= 64 ? 0.55 + 0.0165 * D : 0.0586 * D) * 256 / cu_count();
  return attn_array_ns(tasks * groups, T, D, j) < 5000 + T * std::max(1200.0 + 45.0 * D, tasks * per_task);
}

constexpr int ATTN_GTHREADS = 256;
constexpr int ATTN_DMAX = 2048;  // attn_cpu.cpp:173-174

// One step of a task with S in global memory (Sg = the task's [D][D]) and z
// in LDS: thread j updates the columns it owns (j, j + 256, ...).  q/k/v are
// the step's rows; returns nothing, writes y and (thread 0) den.
__device__ void attn_step_global(float* Sg, float* s_z, float* s_q, float* s_k, float* s_v, float* s_kn,
                                 float* s_inv, const float* q, const float* k, const float* v, float* y,
                                 float* den_out, int D, float eps, float* z_global) {
  const int tid = threadIdx.x;
  for (int i = tid; i < D; i += ATTN_GTHREADS) {
    s_q[i] = q[i];
    s_k[i] = k[i];
    s_v[i] = v[i];
  }
  __syncthreads();
  if (tid == 0) *s_inv = attn_inv_norm(s_k, D);
  __syncthreads();
  const float inv = *s_inv;
  for (int i = tid; i < D; i += ATTN_GTHREADS) {
    const float kn = s_k[i] * inv;
    s_kn[i] = kn;
    const float zi = s_z[i] + kn;
    s_z[i] = zi;
    if (z_global) z_global[i] = zi;
  }
  __syncthreads();
  for (int jj = tid; jj < D; jj += ATTN_GTHREADS) {
    const float vj = s_v[jj];
    float num = 0.0f, den = 0.0f;
    float* col = Sg + jj;
    for (int i = 0; i < D; ++i) {
      const float qi = s_q[i];
      const float sv = col[(int64_t)i * D] + s_kn[i] * vj;
      col[(int64_t)i * D] = sv;
      num = num + qi * sv;
      den = den + qi * s_z[i];
    }
    const float denc = den < eps ? eps : den;
    y[jj] = num / denc;
    if (jj == 0 && den_out) *den_out = denc;
  }
  __syncthreads();  // the LDS rows are rewritten by the next step
}

__global__ void __launch_bounds__(ATTN_GTHREADS)
attn_fwd_global_kernel(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
                       float* __restrict__ Y, float* __restrict__ DEN, float* __restrict__ S_state,
                       float* __restrict__ z_out, int64_t T, int H, int D, float eps) {
  __shared__ float s_q[ATTN_DMAX], s_k[ATTN_DMAX], s_v[ATTN_DMAX], s_kn[ATTN_DMAX], s_z[ATTN_DMAX];
  __shared__ float s_inv;
  const int64_t task = blockIdx.x;
  const int64_t b = task / H, h = task % H;
  const int tid = threadIdx.x;
  float* Sg = S_state + task * D * D;
  // each thread clears the columns it owns; z starts at zero
  for (int jj = tid; jj < D; jj += ATTN_GTHREADS)
    for (int i = 0; i < D; ++i) Sg[(int64_t)i * D + jj] = 0.0f;
  for (int i = tid; i < D; i += ATTN_GTHREADS) s_z[i] = 0.0f;
  __syncthreads();
  const int64_t rs = (int64_t)H * D;
  const int64_t base = (b * T * H + h) * D;
  for (int64_t t = 0; t < T; ++t) {
    const int64_t o = base + t * rs;
    attn_step_global(Sg, s_z, s_q, s_k, s_v, s_kn, &s_inv, Q + o, K + o, V + o, Y + o,
                     DEN ? DEN + (b * T + t) * H + h : nullptr, D, eps, nullptr);
  }
  if (z_out)
    for (int i = tid; i < D; i += ATTN_GTHREADS) z_out[task * D + i] = s_z[i];
}

__global__ void __launch_bounds__(ATTN_GTHREADS)
attn_step_kernel(float* __restrict__ S, float* __restrict__ z, const float* __restrict__ q,
                 const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ y, int D,
                 float eps) {
  __shared__ float s_q[ATTN_DMAX], s_k[ATTN_DMAX], s_v[ATTN_DMAX], s_kn[ATTN_DMAX], s_z[ATTN_DMAX];
  __shared__ float s_inv;
  const int64_t task = blockIdx.x;
  const int64_t o = task * D;
  for (int i = threadIdx.x; i < D; i += ATTN_GTHREADS) s_z[i] = z[o + i];
  __syncthreads();
  attn_step_global(S + task * D * D, s_z, s_q, s_k, s_v, s_kn, &s_inv, q + o, k + o, v + o, y + o, nullptr, D,
                   eps, z + o);
}

// One step for D <= 128: a thread per column, as attn_step_global, but with
// the rows of S in batches of 16 registers, the next batch read before this one
// is updated, so a task waits for D / 16 round trips instead of D, and with
// workgroups of only the waves that have columns.  HBM-bound for many tasks:
// B 64, H 16, D 128 75.7 -> 26.0 us (5.2 TB/s of state read and written), D 64
// 21.4 -> 12.6; a few tasks are the serial sums, 10.2 -> 9.6 us.
template <int NT>
__global__ void __launch_bounds__(NT)
attn_step_col_kernel(float* __restrict__ S, float* __restrict__ z, const float* __restrict__ q,
                     const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ y, int D,
                     float eps) {
  constexpr int NB = 16;
  __shared__ float s_q[NT + NB], s_k[NT], s_kn[NT + NB], s_z[NT + NB];
  __shared__ float s_inv;
  const int64_t task = blockIdx.x, o = task * D;
  const int j = threadIdx.x;
  const bool col = j < D;
  float* Sj = S + task * D * D + (col ? j : D - 1);
  float s[2][NB];
  auto load = [&](auto set, int i0) {  // rows past D: the last one, not used
#pragma unroll
    for (int r = 0; r < NB; ++r) s[set][r] = Sj[(int64_t)(i0 + r < D ? i0 + r : D - 1) * D];
  };
  const float qj = col ? q[o + j] : 0.0f, kj = col ? k[o + j] : 0.0f, vj = col ? v[o + j] : 0.0f;
  const float zj = col ? z[o + j] : 0.0f;
  load(Set<0>(), 0);
  s_k[j] = kj;
  s_q[j] = qj;
  __syncthreads();
  if (j == 0) s_inv = attn_inv_norm(s_k, D);
  __syncthreads();
  const float kn = kj * s_inv, zn = zj + kn;
  s_kn[j] = kn;
  s_z[j] = zn;
  if (col) z[o + j] = zn;
  __syncthreads();
  float num = 0.0f, den = 0.0f;
  auto update = [&](auto set, int i0) {
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      if (i0 + r < D) {  // uniform
        const float qi = s_q[i0 + r];
        const float sv = s[set][r] + s_kn[i0 + r] * vj;
        if (col) Sj[(int64_t)(i0 + r) * D] = sv;
        num = num + qi * sv;
        den = den + qi * s_z[i0 + r];
      }
    }
  };
  for (int i0 = 0; i0 < D; i0 += 2 * NB) {
    load(Set<1>(), i0 + NB);
    update(Set<0>(), i0);
    load(Set<0>(), i0 + 2 * NB);
    update(Set<1>(), i0 + NB);
  }
  const float denc = den < eps ? eps : den;
  if (col) y[o + j] = num / denc;
}

// ---------------------------------------------------------------------------
// backward (attn_cpu.cpp:227-368)
// ---------------------------------------------------------------------------
// Per (b, h) task, two passes over time:
//   A (forward): the recurrence again, then dnum = dy / den, dden = -(dy . y)
//     / den and dq = S dnum + dden z;
//   B (reverse): the adjoints Dm of S and dz of z, Dm += dnum (x) q, dz += dden
//     q, dv = Dm^T kn, dk~ = Dm v + dz, then the key-normalisation backward
//     dk = dk~ / nc - k (k . dk~) / nc^3 (sums in double).
// Bit-identical to the reference kernel: every sum runs in its order.  The
// column sums (num, dv) belong to the thread owning column j and run over i;
// den, (dy . y) and the double sums are sequential, computed by every thread
// that needs them (or thread 0); the row sums (dq, dk~) belong to the thread
// owning row i and run over j the way the reference's 8-lane AVX loop does
// (dot8_lanes).  The state S / Dm is in LDS for D <= 128 (rows padded to D +
// 1 floats, so the row walks of consecutive threads fall in different banks),
// else in the workspace; q/k/v/dy/y are staged CH steps at a time.

// The reference's dot of a row with a vector (attn_cpu.cpp:31-35 and the AVX
// loops feeding hsum8): lane l sums a[j] * b[j] over j = l, l + 8, ... below
// the last multiple of 8, from +0; the lanes are added left to right; the
// remainder follows in order.
__device__ __forceinline__ float dot8_lanes(const float* a, const float* b, int D) {
  float acc[8];
#pragma unroll
  for (int l = 0; l < 8; ++l) acc[l] = 0.0f;
  int j = 0;
  for (; j + 8 <= D; j += 8) {
#pragma unroll
    for (int l = 0; l < 8; ++l) acc[l] = acc[l] + a[j + l] * b[j + l];
  }
  float s = acc[0];
#pragma unroll
  for (int l = 1; l < 8; ++l) s = s + acc[l];
  for (; j < D; ++j) s = s + a[j] * b[j];
  return s;
}

template <int DMAX, int CH, int NT, bool LDS_STATE>
__global__ void __launch_bounds__(NT)
attn_bwd_kernel(const float* __restrict__ dY, const float* __restrict__ Q, const float* __restrict__ K,
                const float* __restrict__ V, const float* __restrict__ Y, const float* __restrict__ DEN,
                float* __restrict__ dQ, float* __restrict__ dK, float* __restrict__ dV, float* __restrict__ state_g,
                int64_t T, int H, int D, float eps) {
  __shared__ float s_state[LDS_STATE ? DMAX * (DMAX + 1) : 1];
  __shared__ float s_q[CH][DMAX], s_k[CH][DMAX], s_v[CH][DMAX], s_dy[CH][DMAX], s_y[CH][DMAX];
  __shared__ float s_kn[DMAX], s_z[DMAX], s_dnum[DMAX], s_t[DMAX];
  __shared__ float s_inv[CH], s_den[CH], s_sc[2];
  const int64_t task = blockIdx.x;
  const int64_t b = task / H, h = task % H;
  const int tid = threadIdx.x;
  float* st = LDS_STATE ? s_state : state_g + task * (int64_t)D * D;
  const int64_t LD = LDS_STATE ? D + 1 : D;
  const int64_t rs = (int64_t)H * D;         // stride between time steps
  const int64_t base = (b * T * H + h) * D;  // (b, t = 0, h)
  auto clear_state = [&]() {
    for (int64_t e = tid; e < (int64_t)D * LD; e += NT) st[e] = 0.0f;
    for (int i = tid; i < D; i += NT) s_z[i] = 0.0f;
  };
  // steps [t0, t0 + nt) of q/k/v/dy (and y, with_y) into the staging rows,
  // their key norms' reciprocals (and DEN) alongside
  auto stage = [&](int64_t t0, int nt, bool with_y) {
    for (int e = tid; e < nt * D; e += NT) {
      const int tt = e / D, j = e - tt * D;
      const int64_t o = base + (t0 + tt) * rs + j;
      s_q[tt][j] = Q[o];
      s_k[tt][j] = K[o];
      s_v[tt][j] = V[o];
      s_dy[tt][j] = dY[o];
      if (with_y) s_y[tt][j] = Y[o];
    }
    __syncthreads();
    for (int tt = tid; tt < nt; tt += NT) {
      s_inv[tt] = attn_inv_norm(s_k[tt], D);
      if (with_y) s_den[tt] = DEN[(b * T + t0 + tt) * H + h];
    }
    __syncthreads();
  };

  // ---- pass A: dQ ----------------------------------------------------------
  clear_state();
  __syncthreads();
  for (int64_t t0 = 0; t0 < T; t0 += CH) {
    const int nt = (int)(T - t0 < CH ? T - t0 : CH);
    stage(t0, nt, false);
    for (int tt = 0; tt < nt; ++tt) {
      const int64_t o = base + (t0 + tt) * rs;
      for (int i = tid; i < D; i += NT) {
        const float kn = s_k[tt][i] * s_inv[tt];
        s_kn[i] = kn;
        s_z[i] = s_z[i] + kn;
      }
      __syncthreads();
      for (int j = tid; j < D; j += NT) {  // column j: S update, num, den
        const float vj = s_v[tt][j];
        float num = 0.0f, den = 0.0f;
        for (int i = 0; i < D; ++i) {
          const float qi = s_q[tt][i];
          const float sv = st[i * LD + j] + s_kn[i] * vj;
          st[i * LD + j] = sv;
          num = num + qi * sv;
          den = den + qi * s_z[i];
        }
        const float denc = den < eps ? eps : den;
        s_t[j] = num / denc;                       // y_j
        s_dnum[j] = s_dy[tt][j] * (1.0f / denc);
        if (j == 0) s_sc[0] = denc;
      }
      __syncthreads();
      const float inv = 1.0f / s_sc[0];
      float yd = 0.0f;
      for (int j = 0; j < D; ++j) yd = yd + s_dy[tt][j] * s_t[j];
      const float dden = -yd * inv;
      for (int i = tid; i < D; i += NT)  // row i: dq
        dQ[o + i] = dot8_lanes(st + i * LD, s_dnum, D) + dden * s_z[i];
      __syncthreads();
    }
  }

  // ---- pass B, reverse in time: dK, dV -----------------------------------
  clear_state();  // Dm and dz
  __syncthreads();
  for (int64_t t1 = T; t1 > 0; t1 -= CH) {
    const int64_t t0 = t1 - CH > 0 ? t1 - CH : 0;
    const int nt = (int)(t1 - t0);
    stage(t0, nt, true);
    for (int tt = nt - 1; tt >= 0; --tt) {
      const int64_t o = base + (t0 + tt) * rs;
      const float invd = 1.0f / s_den[tt];
      for (int i = tid; i < D; i += NT) {
        s_kn[i] = s_k[tt][i] * s_inv[tt];
        s_dnum[i] = s_dy[tt][i] * invd;
      }
      __syncthreads();
      float yd = 0.0f;
      for (int j = 0; j < D; ++j) yd = yd + s_dy[tt][j] * s_y[tt][j];
      const float dden = -yd * invd;
      for (int j = tid; j < D; j += NT) {  // column j: Dm update, dv
        const float dn = s_dnum[j];
        float col = 0.0f;
        for (int i = 0; i < D; ++i) {
          const float dm = st[i * LD + j] + dn * s_q[tt][i];
          st[i * LD + j] = dm;
          col = col + dm * s_kn[i];
        }
        dV[o + j] = col;
      }
      for (int i = tid; i < D; i += NT) s_z[i] = s_z[i] + dden * s_q[tt][i];  // dz
      __syncthreads();
      for (int i = tid; i < D; i += NT) s_t[i] = s_z[i] + dot8_lanes(st + i * LD, s_v[tt], D);  // dk~
      __syncthreads();
      if (tid == 0) {
        double n2 = 0.0, kd = 0.0;
        for (int i = 0; i < D; ++i) {
          const double ki = (double)s_k[tt][i];
          n2 = n2 + ki * ki;
          kd = kd + ki * (double)s_t[i];
        }
        const float n = (float)__builtin_sqrt(n2);
        const float nc = (!__builtin_isfinite(n) || n < 1e-6f) ? 1e-6f : n;
        float sc = (float)(kd / ((double)nc * nc * nc));
        if (!__builtin_isfinite(sc)) sc = 0.0f;
        s_sc[0] = sc;
        s_sc[1] = 1.0f / nc;
      }
      __syncthreads();
      for (int i = tid; i < D; i += NT) dK[o + i] = s_t[i] * s_sc[1] - s_k[tt][i] * s_sc[0];
      __syncthreads();
    }
  }
}

// ---- the backward for D in {16, 32, 48, 64, 96, 128} ------------------------
// The same sums in the same order, spread over four launches:
//  1. attn_bwd_col_kernel: the column passes (sums over i), num / den of pass A
//     and dv of pass B, as the forward's systolic array (attn_col), both in
//     one launch; pass A's y goes to dQ, which is free until step 3.
//  2. attn_bwd_scalars_kernel: per (b, t, h) the serial sums over D: the key
//     norm, dy . y of both passes.
//  3. attn_bwd_row_kernel: the row passes, dq = S dnum + dden z and dk~ = Dm v
//     + dz, again both in one launch.
//  4. attn_bwd_dk_kernel: the key normalisation's backward, in place on dk~.
// One workgroup per task walking 2 T dependent steps (attn_bwd_kernel, which
// the other widths and callers without the workspace keep) takes 5004 us at B
// 8, T 256, H 8, D 64, these four 124 us; at D = 128 (B 8, T 256, H 16) 10340
// and 636 us.  Many short tasks are the other way about (attn_bwd_split).
template <int RPL, int J>
__global__ void __launch_bounds__(AC_NT)
attn_bwd_col_kernel(const float* __restrict__ dY, const float* __restrict__ Q, const float* __restrict__ K,
                    const float* __restrict__ V, const float* __restrict__ DEN, float* __restrict__ Yp,
                    float* __restrict__ DENp, float* __restrict__ dV, int64_t T, int H, int D, int groups, float eps) {
  __shared__ AttnCol<RPL, J> sm;
  if (blockIdx.y == 0)
    attn_col<RPL, J, false>(sm, Q, K, V, nullptr, Yp, DENp, nullptr, nullptr, T, H, D, groups, eps);
  else
    attn_col<RPL, J, true>(sm, Q, K, dY, DEN, dV, nullptr, nullptr, nullptr, T, H, D, groups, eps);
}

// Per row r = (b, t, h), each [rows]: inv = 1 / max(||k||, 1e-6); 1 / den and
// -(dy . y) / den of pass A (its own y and den) and of pass B (the caller's).
struct BwdScalars {
  float *inv, *invA, *ddenA, *invB, *ddenB;
};

template <int DMAX>
__global__ void __launch_bounds__(192)
attn_bwd_scalars_kernel(const float* __restrict__ K, const float* __restrict__ dY, const float* __restrict__ Yp,
                        const float* __restrict__ Y, const float* __restrict__ DENp, const float* __restrict__ DEN,
                        BwdScalars o, int64_t rows, int D) {
  __shared__ float sm[4][64 * (DMAX + 1)];
  const int64_t r0 = (int64_t)blockIdx.x * 64;
  const int nr = (int)(rows - r0 < 64 ? rows - r0 : 64);
  for (int e = threadIdx.x; e < nr * D; e += 192) {
    const int r = e / D, j = e - r * D, d = r * (D + 1) + j;
    const int64_t g = r0 * D + e;
    sm[0][d] = K[g];
    sm[1][d] = dY[g];
    sm[2][d] = Yp[g];
    sm[3][d] = Y[g];
  }
  __syncthreads();
  const int what = threadIdx.x >> 6, r = threadIdx.x & 63;
  if (r >= nr) return;
  if (what == 0) {
    o.inv[r0 + r] = attn_inv_norm(sm[0] + r * (D + 1), D);
    return;
  }
  const float *dy = sm[1] + r * (D + 1), *y = sm[1 + what] + r * (D + 1);
  float yd = 0.0f;
  for (int j = 0; j < D; ++j) yd = yd + dy[j] * y[j];
  const float inv = 1.0f / (what == 1 ? DENp : DEN)[r0 + r];
  (what == 1 ? o.invA : o.invB)[r0 + r] = inv;
  (what == 1 ? o.ddenA : o.ddenB)[r0 + r] = -yd * inv;
}

// dk = dk~ / nc - k (k . dk~) / nc^3 per row, dK holding dk~ (sums in double).
template <int DMAX>
__global__ void __launch_bounds__(256)
attn_bwd_dk_kernel(const float* __restrict__ K, float* __restrict__ dK, int64_t rows, int D) {
  __shared__ float sk[64 * (DMAX + 1)], st[64 * (DMAX + 1)];
  __shared__ float s_inv[64], s_sc[64];
  const int64_t r0 = (int64_t)blockIdx.x * 64;
  const int nr = (int)(rows - r0 < 64 ? rows - r0 : 64);
  for (int e = threadIdx.x; e < nr * D; e += 256) {
    const int r = e / D, d = e + r;  // rows of D + 1
    sk[d] = K[r0 * D + e];
    st[d] = dK[r0 * D + e];
  }
  __syncthreads();
  const int r = threadIdx.x;
  if (r < nr) {
    double n2 = 0.0, kd = 0.0;
    for (int i = 0; i < D; ++i) {
      const double ki = (double)sk[r * (D + 1) + i];
      n2 = n2 + ki * ki;
      kd = kd + ki * (double)st[r * (D + 1) + i];
    }
    const float n = (float)__builtin_sqrt(n2);
    const float nc = (!__builtin_isfinite(n) || n < 1e-6f) ? 1e-6f : n;
    float sc = (float)(kd / ((double)nc * nc * nc));
    if (!__builtin_isfinite(sc)) sc = 0.0f;
    s_sc[r] = sc;
    s_inv[r] = 1.0f / nc;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nr * D; e += 256) {
    const int rr = e / D, d = e + rr;
    dK[r0 * D + e] = st[d] * s_inv[rr] - sk[d] * s_sc[rr];
  }
}

// The row passes: row i of the state belongs to 8 lanes, lane l of them to its
// columns l, l + 8, ... (the 8 partial sums of dot8_lanes), M = D / 8 of them
// in registers.  The partials are added left to right by moving the running
// sum one lane on per tick (row_shr:1 on the add), so lane l works on step t =
// tau - l and lane 7 finishes a step every tick.  Pass A: state S += kn (x) v,
// dq = S dnum + dden z; pass B (REV, time backwards): Dm += q (x) dnum, dk~ =
// Dm v + dz.  A workgroup is 4 computing waves (8 rows each) and one that
// stages the next 16 steps into a ring of 64.
//
// What bounds it: LDS reads (4 of 16 bytes per tick and wave for M = 8, all
// rows reading the same 8 lanes' columns) about level with the 4 M VALU
// operations per tick, on 2 B H D / 32 workgroups of both passes together.
constexpr int AR_W = 4, AR_NT = (AR_W + 1) * 64, AR_CH = 16, AR_RN = 64, AR_ROWS = AR_W * 8;

template <int M>
struct AttnRow {
  static constexpr int DP = (8 * M + 63) / 64;  // columns of a staging lane
  // b [l][m], c [l][m], a (the rows), dden; padded so that the 8 lanes' reads,
  // one ring row apart, fall in different banks
  static constexpr int RB = 16 * M + (M % 8 == 4 ? 40 : 36);
  static constexpr int NB = M <= 8 ? 4 : 2;     // ticks whose operands are read together
  __attribute__((aligned(16))) float row[AR_RN * RB];
};

template <int M>
__device__ __forceinline__ void attn_read_cols(const float* p, float (&d)[M]) {
  if constexpr (M % 4 == 0) {
#pragma unroll
    for (int m = 0; m < M; m += 4) {
      const float4 w = *(const float4*)(p + m);
      d[m] = w.x;
      d[m + 1] = w.y;
      d[m + 2] = w.z;
      d[m + 3] = w.w;
    }
  } else {
#pragma unroll
    for (int m = 0; m < M; m += 2) {
      const float2 w = *(const float2*)(p + m);
      d[m] = w.x;
      d[m + 1] = w.y;
    }
  }
}

template <int M, bool REV>
__device__ __forceinline__ void
attn_row(AttnRow<M>& sm, const float* __restrict__ dY, const float* __restrict__ Q, const float* __restrict__ K,
         const float* __restrict__ V, const BwdScalars& sc, float* __restrict__ out, int64_t T, int H, int groups) {
  using L = AttnRow<M>;
  constexpr int D = 8 * M, RB = L::RB, DP = L::DP, NB = L::NB, CH = AR_CH;
  const int64_t task = blockIdx.x / groups;
  const int i0 = (int)(blockIdx.x - task * groups) * AR_ROWS;
  const int64_t b = task / H, h = task % H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t hs = REV ? -H : H;                            // stride between steps, in rows of D
  const int64_t base = (b * T + (REV ? T - 1 : 0)) * H + h;   // and the first one
  const int64_t chunks = (T + 7 + CH - 1) / CH;

  for (int e = tid; e < AR_RN * RB; e += AR_NT) sm.row[e] = 0.0f;

  if (wave == AR_W) {
    constexpr int AN = CH * AR_ROWS / 64;
    const float* A = REV ? Q : K;
    float sv[2][CH * DP], sg[2][CH * DP], sa[2][AN], s1[2], s2[2], s3[2];
    uint32_t col[DP];
#pragma unroll
    for (int p = 0; p < DP; ++p) col[p] = lane + 64 * p < D ? lane + 64 * p : D - 1;
    const int ai = i0 + (lane & 31) < D ? i0 + (lane & 31) : D - 1;
    auto load = [&](auto set, int64_t c) {
      const int64_t left = T - c * CH;
      const int64_t row = base + (left > 0 ? c * CH : 0) * hs;
      int64_t o = row;
#pragma unroll
      for (int r = 0; r < CH; ++r) {  // steps past T: the last one again, cleared when staged
#pragma unroll
        for (int p = 0; p < DP; ++p) {
          sv[set][r * DP + p] = V[o * D + col[p]];
          sg[set][r * DP + p] = dY[o * D + col[p]];
        }
        o += r + 1 < left ? hs : 0;
      }
#pragma unroll
      for (int n = 0; n < AN; ++n) {
        const int r = 2 * n + (lane >> 5);
        sa[set][n] = A[(row + (r < left ? r : 0) * hs) * D + ai];
      }
      const int64_t rr = row + ((lane & (CH - 1)) < left ? lane & (CH - 1) : 0) * hs;
      s1[set] = REV ? sc.invB[rr] : sc.invA[rr];
      s2[set] = REV ? sc.ddenB[rr] : sc.ddenA[rr];
      if constexpr (!REV) s3[set] = sc.inv[rr];
    };
    auto stage = [&](auto set, int64_t c) {
      const int64_t left = T - c * CH;
      float* rows = sm.row + (int)(c % (AR_RN / CH)) * CH * RB;
#pragma unroll
      for (int r = 0; r < CH; ++r) {
        const float invd = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s1[set]), r));
#pragma unroll
        for (int p = 0; p < DP; ++p) {
          const int j = lane + 64 * p;
          const float v = r < left ? sv[set][r * DP + p] : 0.0f;
          const float dn = r < left ? sg[set][r * DP + p] * invd : 0.0f;
          if (DP * 64 == D || j < D) {
            rows[r * RB + (j & 7) * M + (j >> 3)] = REV ? dn : v;
            rows[r * RB + 8 * M + (j & 7) * M + (j >> 3)] = REV ? v : dn;
          }
        }
      }
#pragma unroll
      for (int n = 0; n < AN; ++n) {
        const int r = 2 * n + (lane >> 5);
        float a = sa[set][n];
        if constexpr (!REV) a = a * __shfl(s3[set], r, 64);
        rows[r * RB + 16 * M + (lane & 31)] = r < left ? a : 0.0f;
      }
      if (lane < CH) rows[lane * RB + 16 * M + AR_ROWS] = lane < left ? s2[set] : 0.0f;
    };
    load(Set<0>(), 0);
    load(Set<1>(), 1);
    __syncthreads();
    stage(Set<0>(), 0);
    load(Set<0>(), 2);
    __syncthreads();
    for (int64_t c = 0; c < chunks; c += 2) {  // period c stages chunk c + 1
      if (c + 1 < chunks) {
        stage(Set<1>(), c + 1);
        load(Set<1>(), c + 3);
      }
      __syncthreads();
      if (c + 1 < chunks) {
        if (c + 2 < chunks) {
          stage(Set<0>(), c + 2);
          load(Set<0>(), c + 4);
        }
        __syncthreads();
      }
    }
    return;
  }

  const int l = lane & 7, ri = wave * 8 + (lane >> 3), i = i0 + ri;
  float S[M], z = 0.0f, s = 0.0f;
#pragma unroll
  for (int m = 0; m < M; ++m) S[m] = 0.0f;
  const bool writes = l == 7 && i < D;
  float* op = out + (base - 7 * hs) * D + i;  // lane 7's step at tick 0 is -7
  __syncthreads();
  __syncthreads();
  int64_t tau = 0;
  for (int64_t c = 0; c < chunks; ++c) {
    const int tick0 = (int)(c % (AR_RN / CH)) * CH;
    float bb[2][NB][M], cc[2][NB][M], aa[2][NB], dd[2][NB];
    auto fetch = [&](int set, int tt, int tick) {
      const float* p = sm.row + ((tick0 + tick - l) & (AR_RN - 1)) * RB;
      attn_read_cols<M>(p + l * M, bb[set][tt]);
      attn_read_cols<M>(p + 8 * M + l * M, cc[set][tt]);
      aa[set][tt] = p[16 * M + ri];
      dd[set][tt] = p[16 * M + AR_ROWS];
    };
#pragma unroll
    for (int tt = 0; tt < NB; ++tt) fetch(0, tt, tt);
#pragma unroll
    for (int tt0 = 0; tt0 < CH; tt0 += NB) {
      const int g = (tt0 / NB) & 1;
#pragma unroll
      for (int tt = 0; tt < NB; ++tt) {
        if (tt0 + NB < CH) fetch(g ^ 1, tt, tt0 + NB + tt);
        const float a = aa[g][tt];
        float acc = 0.0f;
#pragma unroll
        for (int m = 0; m < M; ++m) {
          S[m] = S[m] + a * bb[g][tt][m];
          acc = acc + S[m] * cc[g][tt][m];
        }
        // lane 0 of the 8 starts the sum
        const float before = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x111, 0xf, 0xf, true));
        s = l == 0 ? acc : before + acc;
        float r;
        if constexpr (REV) {
          z = z + dd[g][tt] * a;
          r = z + s;
        } else {
          z = z + a;
          r = s + dd[g][tt] * z;
        }
        if (writes && tau >= 7 && tau < T + 7) *op = r;
        op += hs * D;
        ++tau;
      }
    }
    __syncthreads();
  }
}

template <int M>
__global__ void __launch_bounds__(AR_NT)
attn_bwd_row_kernel(const float* __restrict__ dY, const float* __restrict__ Q, const float* __restrict__ K,
                    const float* __restrict__ V, BwdScalars sc, float* __restrict__ dQ, float* __restrict__ dK,
                    int64_t T, int H, int groups) {
  __shared__ AttnRow<M> sm;
  if (blockIdx.y == 0)
    attn_row<M, false>(sm, dY, Q, K, V, sc, dQ, T, H, groups);
  else
    attn_row<M, true>(sm, dY, Q, K, V, sc, dK, T, H, groups);
}

// Whether a backward runs as the four launches: a head width that the row pass is
// instantiated for (whole 8-lane rows, and an even M for its vector reads; the
// other widths run attn_bwd_kernel), and the sooner end
// of the two from what they measure, in ns: 15000 and both column passes, and
// per task and 32 rows of the row passes 45 and, a step, 0.8 + 0.0095 D (one
// task alone 2.5 D), against attn_bwd_kernel's steps of 1200 + 300 D, or of a time
// per task where the CUs are full.  us, four / one:
//   D 64   T 1: 8 tasks 27 / 29, 512 202 / 31, 16384 5814 / 468    T 4: 128 tasks 77 / 87
//   D 64  T 16: 128 tasks 81 / 318, 512 262 / 326, 2048 985 / 683, 16384 7812 / 5499
//   D 64  T 64: 2048 tasks 1393 / 2704
//   D 128  T 4: 128 tasks 171 / 176, 512 581 / 351, 16384 17468 / 11003    T 16: 16384 tasks 19606 / 41708
//   D 16   T 4: 8 tasks 23 / 28, 512 80 / 28    T 16: 512 tasks 88 / 98, 2048 318 / 203    T 64: 2048 564 / 809
bool attn_bwd_split(int64_t tasks, int64_t T, int64_t D) {
  if (!(D == 16 || D == 32 || D == 48 || D == 64 || D == 96 || D == 128)) return false;
  const int j = attn_col_width(2 * tasks, D);
  const int64_t groups = (D + AC_W * j - 1) / (AC_W * j), rgroups = (D + AR_ROWS - 1) / AR_ROWS;
  if (tasks * groups >= ATTN_GRID_THREADS / AC_NT || tasks * rgroups >= ATTN_GRID_THREADS / AR_NT) return false;
  const double full = 256.0 / cu_count();
  const double rows = std::max(2.5 * D * T, tasks * rgroups * (45 + T * (0.8 + 0.0095 * D)) * full);
  const double step = std::max(1200.0 + 300.0 * D, tasks * (D <= 64 ? 0.9 + 0.31 * D : 1.23 * D) * full);
  return 15000 + attn_array_ns(2 * tasks * groups, T, D, j) + rows < 5000 + T * step;
}

int attn_bwd_launch(const float* dY, const float* Q, const float* K, const float* V, const float* Y, const float* DEN,
                    float* dQ, float* dK, float* dV, int64_t B, int64_t T, int64_t H, int64_t D, float eps, float* ws,
                    hipStream_t stream) {
  const int64_t rows = B * T * H;
  const BwdScalars sc = {ws + rows, ws + 2 * rows, ws + 3 * rows, ws + 4 * rows, ws + 5 * rows};
  const int j = attn_col_width(2 * B * H, D);
  const int64_t groups = (D + AC_W * j - 1) / (AC_W * j);
  auto col = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(B * H * groups), 2), dim3(AC_NT), 0, stream, dY, Q, K, V, DEN, dQ, ws,
                       dV, T, (int)H, (int)D, (int)groups, eps);
  };
  if (D <= 64)
    j == 2 ? col(attn_bwd_col_kernel<1, 2>) : j == 4 ? col(attn_bwd_col_kernel<1, 4>) : col(attn_bwd_col_kernel<1, 8>);
  else
    j == 2 ? col(attn_bwd_col_kernel<2, 2>) : j == 4 ? col(attn_bwd_col_kernel<2, 4>) : col(attn_bwd_col_kernel<2, 8>);
  int rc = check_launch("attn_bwd_col_kernel");
  if (rc) return rc;
  const dim3 rgrid((unsigned)((rows + 63) / 64));
  if (D <= 64)
    hipLaunchKernelGGL((attn_bwd_scalars_kernel<64>), rgrid, dim3(192), 0, stream, K, dY, dQ, Y, ws, DEN, sc, rows,
                       (int)D);
  else
    hipLaunchKernelGGL((attn_bwd_scalars_kernel<128>), rgrid, dim3(192), 0, stream, K, dY, dQ, Y, ws, DEN, sc, rows,
                       (int)D);
  rc = check_launch("attn_bwd_scalars_kernel");
  if (rc) return rc;
  const int64_t rgroups = (D + AR_ROWS - 1) / AR_ROWS;
  auto row = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(B * H * rgroups), 2), dim3(AR_NT), 0, stream, dY, Q, K, V, sc, dQ, dK,
                       T, (int)H, (int)rgroups);
  };
  switch (D) {
    case 16: row(attn_bwd_row_kernel<2>); break;
    case 32: row(attn_bwd_row_kernel<4>); break;
    case 48: row(attn_bwd_row_kernel<6>); break;
    case 64: row(attn_bwd_row_kernel<8>); break;
    case 96: row(attn_bwd_row_kernel<12>); break;
    default: row(attn_bwd_row_kernel<16>); break;
  }
  rc = check_launch("attn_bwd_row_kernel");
  if (rc) return rc;
  if (D <= 64)
    hipLaunchKernelGGL((attn_bwd_dk_kernel<64>), rgrid, dim3(256), 0, stream, K, dK, rows, (int)D);
  else
    hipLaunchKernelGGL((attn_bwd_dk_kernel<128>), rgrid, dim3(256), 0, stream, K, dK, rows, (int)D);
  return check_launch("attn_bwd_dk_kernel");
}

int check_attn_shape(int64_t B, int64_t T, int64_t H, int64_t D, float eps, const char* what) {
  if (B < 0 || T < 0 || H < 0 || D <= 0)
    return fail(SMAUL_ERR_INVALID, "%s: bad shape [%lld,%lld,%lld,%lld]", what, (long long)B, (long long)T,
                (long long)H, (long long)D);
  if (D > ATTN_DMAX)
    return fail(SMAUL_ERR_INVALID, "%s: D=%lld out of the supported range (0, %d]", what, (long long)D, ATTN_DMAX);
  if (!(eps > 0.0f) || !__builtin_isfinite(eps))
    return fail(SMAUL_ERR_INVALID, "%s: eps must be positive finite, got %g", what, (double)eps);
  if (B * H > 2147483647LL) return fail(SMAUL_ERR_UNSUPPORTED, "%s: B*H exceeds the grid", what);
  if (H > 2147483647LL) return fail(SMAUL_ERR_UNSUPPORTED, "%s: H too large", what);
  return SMAUL_OK;
}

}  // namespace

extern "C" {

int64_t smaul_attn_workspace_size(int64_t B, int64_t H, int64_t D, int need_state) {
  if (B < 0 || H < 0 || D <= 0) return -1;
  if (D <= 128 || need_state) return 0;
  return B * H * D * D * (int64_t)sizeof(float);
}

int64_t smaul_attn_backward_workspace_size(int64_t B, int64_t T, int64_t H, int64_t D) {
  if (B < 0 || T < 0 || H < 0 || D <= 0) return -1;
  if (attn_bwd_split(B * H, T, D)) return 6 * B * T * H * (int64_t)sizeof(float);
  return smaul_attn_workspace_size(B, H, D, 0);
}

int smaul_attn_forward(const float* Q, const float* K, const float* V, float* Y, float* DEN, float* S_out,
                       float* z_out, int64_t B, int64_t T, int64_t H, int64_t D, float eps, void* workspace,
                       int64_t workspace_bytes, hipStream_t stream) {
  int rc = check_attn_shape(B, T, H, D, eps, "attn_forward");
  if (rc) return rc;
  if ((S_out == nullptr) != (z_out == nullptr))
    return fail(SMAUL_ERR_INVALID, "attn_forward: S_out and z_out go together");
  if (B == 0 || H == 0) return SMAUL_OK;
  if (T > 0 && (!Q || !K || !V || !Y)) return fail(SMAUL_ERR_INVALID, "attn_forward: null pointer");
  const dim3 grid((unsigned)(B * H));
  if (D <= 128) {
    if (T == 0 && !S_out) return SMAUL_OK;  // T == 0 with a state: the kernel writes zeros
    const int j = attn_col_width(B * H, D);
    const int64_t groups = (D + AC_W * j - 1) / (AC_W * j);
    if (!attn_use_array(B * H, T, D, j, groups)) {
      if (D <= 64)
        hipLaunchKernelGGL((attn_fwd_reg_kernel<64>), grid, dim3(64), 0, stream, Q, K, V, Y, DEN, S_out, z_out, T,
                           (int)H, (int)D, eps);
      else
        hipLaunchKernelGGL((attn_fwd_reg_kernel<128>), grid, dim3(128), 0, stream, Q, K, V, Y, DEN, S_out, z_out, T,
                           (int)H, (int)D, eps);
      return check_launch("attn_fwd_reg_kernel");
    }
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(B * H * groups)), dim3(AC_NT), 0, stream, Q, K, V, Y, DEN, S_out,
                         z_out, T, (int)H, (int)D, (int)groups, eps);
    };
    if (D <= 64)
      j == 2 ? go(attn_fwd_col_kernel<1, 2>) : j == 4 ? go(attn_fwd_col_kernel<1, 4>) : go(attn_fwd_col_kernel<1, 8>);
    else
      j == 2 ? go(attn_fwd_col_kernel<2, 2>) : j == 4 ? go(attn_fwd_col_kernel<2, 4>) : go(attn_fwd_col_kernel<2, 8>);
    return check_launch("attn_fwd_col_kernel");
  }
  float* state = S_out;
  if (!state) {
    const int64_t need = smaul_attn_workspace_size(B, H, D, 0);
    if (workspace_bytes < need || !workspace)
      return fail(SMAUL_ERR_INVALID, "attn_forward: workspace %lld < %lld bytes", (long long)workspace_bytes,
                  (long long)need);
    state = (float*)workspace;
  }
  if (T == 0 && !S_out) return SMAUL_OK;
  hipLaunchKernelGGL(attn_fwd_global_kernel, grid, dim3(ATTN_GTHREADS), 0, stream, Q, K, V, Y, DEN, state, z_out, T,
                     (int)H, (int)D, eps);
  return check_launch("attn_fwd_global_kernel");
}

int smaul_attn_step(float* S, float* z, const float* q, const float* k, const float* v, float* y, int64_t B,
                    int64_t H, int64_t D, float eps, hipStream_t stream) {
  int rc = check_attn_shape(B, 1, H, D, eps, "attn_step");
  if (rc) return rc;
  if (B == 0 || H == 0) return SMAUL_OK;
  if (!S || !z || !q || !k || !v || !y) return fail(SMAUL_ERR_INVALID, "attn_step: null pointer");
  const dim3 grid((unsigned)(B * H));
  if (D <= 64)
    hipLaunchKernelGGL((attn_step_col_kernel<64>), grid, dim3(64), 0, stream, S, z, q, k, v, y, (int)D, eps);
  else if (D <= 128)
    hipLaunchKernelGGL((attn_step_col_kernel<128>), grid, dim3(128), 0, stream, S, z, q, k, v, y, (int)D, eps);
  else
    hipLaunchKernelGGL(attn_step_kernel, grid, dim3(ATTN_GTHREADS), 0, stream, S, z, q, k, v, y, (int)D, eps);
  return check_launch("attn_step_kernel");
}

int smaul_attn_backward(const float* dY, const float* Q, const float* K, const float* V, const float* Y,
                        const float* DEN, float* dQ, float* dK, float* dV, int64_t B, int64_t T, int64_t H, int64_t D,
                        float eps, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  int rc = check_attn_shape(B, T, H, D, eps, "attn_backward");
  if (rc) return rc;
  if (B == 0 || H == 0 || T == 0) return SMAUL_OK;
  if (!dY || !Q || !K || !V || !Y || !DEN || !dQ || !dK || !dV)
    return fail(SMAUL_ERR_INVALID, "attn_backward: null pointer");
  if (attn_bwd_split(B * H, T, D) && workspace && workspace_bytes >= smaul_attn_backward_workspace_size(B, T, H, D))
    return attn_bwd_launch(dY, Q, K, V, Y, DEN, dQ, dK, dV, B, T, H, D, eps, (float*)workspace, stream);
  const dim3 grid((unsigned)(B * H));
  if (D <= 64) {
    hipLaunchKernelGGL((attn_bwd_kernel<64, 16, 64, true>), grid, dim3(64), 0, stream, dY, Q, K, V, Y, DEN, dQ, dK,
                       dV, nullptr, T, (int)H, (int)D, eps);
    return check_launch("attn_bwd_kernel");
  }
  if (D <= 128) {
    hipLaunchKernelGGL((attn_bwd_kernel<128, 16, 128, true>), grid, dim3(128), 0, stream, dY, Q, K, V, Y, DEN, dQ,
                       dK, dV, nullptr, T, (int)H, (int)D, eps);
    return check_launch("attn_bwd_kernel");
  }
  const int64_t need = smaul_attn_workspace_size(B, H, D, 0);
  if (workspace_bytes < need || !workspace)
    return fail(SMAUL_ERR_INVALID, "attn_backward: workspace %lld < %lld bytes", (long long)workspace_bytes,
                (long long)need);
  hipLaunchKernelGGL((attn_bwd_kernel<ATTN_DMAX, 1, ATTN_GTHREADS, false>), grid, dim3(ATTN_GTHREADS), 0, stream, dY,
                     Q, K, V, Y, DEN, dQ, dK, dV, (float*)workspace, T, (int)H, (int)D, eps);
  return check_launch("attn_bwd_kernel");
}

}  // extern "C"
