// DropKV scoring on the matrix cores for the inputs outside the tuned
// pipeline of dkv_score.hip: fp32 Q/K/V of head dimensions up to 256, and
// bf16 / fp16 ones of head dimensions other than 32, 64 and 128 (80, 96, 192,
// 256, ...).  Same semantics and at least the precision of the vector-ALU
// kernels in dkv_generic.hip, which keep the head dimensions these do not
// take (above 256, or rows that are no whole 16-byte units).
//
// Nothing is rounded that those kernels keep in fp32:
//   * logits: products of the inputs summed in fp32 (the bf16 / fp16 matrix
//     instructions for 16-bit inputs, whose products are exact, the fp32 one,
//     v_mfma_f32_16x16x4_f32, otherwise), the same sum in every kernel;
//   * p = 2^((logit - row maximum) / ln 2) / row sum, the difference taken of
//     the unscaled logits (exactly 0 at the maximum, however large it is), from the same two numbers wherever
//     it is used.  Where a key takes nearly all of a row's attention, its score
//     (p / (1 - p))^2 |v - y|^2 holds 1 - p twice, once in y: an error of p
//     cancels if both come from the same p (with the logarithm of the sum,
//     whose own rounding is a relative error of p, in between, such scores
//     were up to 20 times further from the 64-bit ones);
//   * y = sum_j p_j v_j with the final p, rounded to the input type first
//     when p_round (then a sweep for the log-sum-exp comes before), fp32
//     products and sums;
//   * |v - y|^2 as |v|^2 - 2<v,y> + |y|^2 with <v,y> from fp32 operands (or
//     from y in the input type where y was rounded to it: the same value),
//     and taken directly, element by element, wherever that sum cancels to
//     less than a quarter of its terms.
//
// What bounds them: at the sizes these inputs are used at (a few thousand
// keys), latency: three or four launches, and in each one round trip to memory
// for the operands, the matrix instructions of a tile and a reduction.  The
// vector-ALU kernels read K with one row per lane (16 lanes of a load in 16
// different rows) and gave each query row a workgroup of its own: 3990 us for
// 8192 keys of D 256 in bf16 (8 query, 4 KV heads), 3650 us for 8192 keys of D
// 64 in fp32 (14, 2), 1790 us for 4099 keys of D 96 in fp16 (16, 16); these
// kernels take 49, 34 and 34 us.
//
// Kernels (fp32 inputs, or no p rounding: 1, 3, 4; else 1, 2, 3, 4):
//   1. part<kFlash>: per (head, 32 query rows, key split) the row maxima, sums
//      and unnormalised y of an online softmax; part<kStats>: maxima and sums;
//   2. part<kSum>: y of the split with the final, rounded p;
//   3. merge: one wave per row: maximum and sum, y, |y|^2;
//   4. score: per key the sum over the rows.
#include "dkv_common.h"
#include "dkv_internal.h"

#include <algorithm>

namespace dkv {

namespace {

constexpr int kRowsC = 32;        // query rows per chunk (the plan's partial layout)
constexpr int kPartWaves = 8;     // waves of a part workgroup
constexpr int kPartKeys = 256;    // keys per step of a part workgroup: 32 per wave
constexpr int kPPitch = kPartKeys + 4;  // floats per row of P in LDS
constexpr int kScoreWaves = 4;
constexpr float kDirect = 0.25f;  // dist2 below this share of its terms is taken directly

// Chunks whose loads a wave issues together (those past D are no request).
constexpr int kGrp = 8;

enum { kStats = 0, kSum = 1, kFlash = 2 };

// Elements per 16 bytes, and the head-dim columns that one 16-byte load per
// lane covers of 16 rows (4 lane groups x 16 bytes).
template <typename T>
constexpr int kEpl = 16 / (int)sizeof(T);
template <typename T>
constexpr int kCols = 4 * kEpl<T>;

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ float elem_of(u32x4 x, int e);
template <>
__device__ __forceinline__ float elem_of<float>(u32x4 x, int e) {
  return __uint_as_float(x[e]);
}
template <>
__device__ __forceinline__ float elem_of<__bf16>(u32x4 x, int e) {
  return __uint_as_float((e & 1) ? (x[e / 2] & 0xffff0000u) : (x[e / 2] << 16));
}
template <>
__device__ __forceinline__ float elem_of<_Float16>(u32x4 x, int e) {
  return static_cast<float>(__builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? (x[e / 2] >> 16) : (x[e / 2] & 0xffffu))));
}

// c += A B over the kCols<T> columns of one chunk: lane (li, lg) holds columns
// kEpl * lg .. of row li of A and of row li of B.
template <typename T>
__device__ __forceinline__ f32x4 mfma_chunk(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (sizeof(T) == 2) {
    typedef typename Elem<T>::v8 v8;
    return Elem<T>::mfma(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = mfma_f32(__uint_as_float(a[e]), __uint_as_float(b[e]), c);
    return c;
  }
}

// Four consecutive elements at byte offset `off` as floats.
template <typename T>
__device__ __forceinline__ f32x4 load4(rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  } else {
    const i32x2 x = buf_load8i(r, off);
    const u32x4 w = {(uint32_t)x[0], (uint32_t)x[1], 0u, 0u};
    return f32x4{elem_of<T>(w, 0), elem_of<T>(w, 1), elem_of<T>(w, 2), elem_of<T>(w, 3)};
  }
}

constexpr uint32_t kPastAll = 0xfffffff0u;  // an offset past every view: zeros, no memory request

// Query rows m0 .. m0 + 16 * kRB - 1 as MFMA operands in LDS: slot (rb, chunk,
// lane) holds the lane's 16 bytes; zeros past row M and column D.
template <typename T, int kRB, int NT>
__device__ __forceinline__ void stage_q(u32x4* qop, int nch, const T* __restrict__ q, int64_t q_sb, int64_t q_sh,
                                        int64_t q_ss, int64_t q_sd, int b, int hkv, int g, int W, int Lq, int M,
                                        int D, int m0) {
  for (int s = threadIdx.x; s < kRB * nch * 64; s += NT) {
    const int lane = s & 63, c = (s >> 6) % nch, rb = (s >> 6) / nch;
    const int m = m0 + 16 * rb + (lane & 15), d0 = c * kCols<T> + kEpl<T> * (lane >> 4);
    T x[kEpl<T>];
    const int mm = min(m, M - 1);
    const T* row = q + (int64_t)b * q_sb + (int64_t)(hkv * g + mm / W) * q_sh + (int64_t)(Lq - W + mm % W) * q_ss;
#pragma unroll
    for (int e = 0; e < kEpl<T>; ++e) x[e] = row[(int64_t)min(d0 + e, D - 1) * q_sd];
#pragma unroll
    for (int e = 0; e < kEpl<T>; ++e)
      if (m >= M || d0 + e >= D) x[e] = static_cast<T>(0.f);
    u32x4 w;
    __builtin_memcpy(&w, x, 16);
    qop[s] = w;
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// One workgroup per (head, 32-row chunk, key split), in steps of 256 keys: each
// wave takes 32 of them for the logits (S^T = K Q^T: a lane holds one query row
// and four keys per block, so row maxima and sums are mostly in-lane), the
// probabilities go to LDS as fp32, and for Y^T += V^T P^T the waves share the
// step's keys and the head dimension: 64 columns and 256 / KG keys each, so
// that V comes straight from memory in the operand's layout (a lane's four
// consecutive columns feed four MFMAs, one per column).  The KG partial sums
// are added in LDS in a fixed order.
// ---------------------------------------------------------------------------
template <typename T, int kRB, int kMode>
__global__ void __launch_bounds__(64 * kPartWaves)
genm_part_kernel(const T* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_sd,
                 const T* __restrict__ kp, const T* __restrict__ vp, KvStride kvs, int Hkv, int Lq, int Lk, int D,
                 int W, int g, int M, int n_mc, int n_splits, int kps, float scale_log2,
                 float* __restrict__ part_ml, float* __restrict__ part_y, float* __restrict__ row_mr) {
  constexpr int NT = 64 * kPartWaves;
  constexpr int R = 16 * kRB;
  extern __shared__ u32x4 gm_lds[];
  __shared__ float wred[2][kPartWaves][kRowsC];
  __shared__ float row_m[kRowsC], row_r[kRowsC];  // kSum: the rows' maxima and 1 / sums
  const int nch = (D + kCols<T> - 1) / kCols<T>;
  u32x4* qop = gm_lds;
  float* P = reinterpret_cast<float*>(qop + kRB * nch * 64);

  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int mc = lid % n_mc, split = (lid / n_mc) % n_splits, head = lid / (n_mc * n_splits);
  const int b = head / Hkv, hkv = head % Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int k_begin = split * kps, k_end = min(k_begin + kps, Lk), nrel = k_end - k_begin;
  const rsrc_t krs = make_rsrc(reinterpret_cast<const char*>(kp + b * kvs.k_sb + hkv * kvs.k_sh) +
                                   (int64_t)k_begin * kvs.k_rb,
                               rows_bytes(nrel, kvs.k_rb, D * (uint32_t)sizeof(T)));
  const rsrc_t vrs = make_rsrc(reinterpret_cast<const char*>(vp + b * kvs.v_sb + hkv * kvs.v_sh) +
                                   (int64_t)k_begin * kvs.v_rb,
                               rows_bytes(nrel, kvs.v_rb, D * (uint32_t)sizeof(T)));
  const int64_t slot = ((int64_t)head * n_mc + mc) * n_splits + split;

  stage_q<T, kRB, NT>(qop, nch, q, q_sb, q_sh, q_ss, q_sd, b, hkv, g, W, Lq, M, D, mc * kRowsC);
  if constexpr (kMode == kSum) {
    // The rows' log-sum-exp from the splits' maxima and sums: 16 threads a row.
    const int row = tid >> 4;
    const float* ml = part_ml + (((int64_t)head * n_mc + mc) * n_splits) * kRowsC * 2;
    float mx = -INFINITY;
    for (int s = tid & 15; s < n_splits; s += 16) mx = fmaxf(mx, ml[(s * kRowsC + row) * 2]);
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    float l = 0.f;
    for (int s = tid & 15; s < n_splits; s += 16) {
      const float m = ml[(s * kRowsC + row) * 2];
      if (m != -INFINITY) l += ml[(s * kRowsC + row) * 2 + 1] * exp2f((m - mx) * scale_log2);
    }
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) l += __shfl_xor(l, o);
    if ((tid & 15) == 0) {
      row_m[row] = mx;
      row_r[row] = 1.f / l;
      if (split == 0 && row < R)
        reinterpret_cast<float2*>(row_mr)[((int64_t)head * n_mc + mc) * kRowsC + row] = make_float2(mx, 1.f / l);
    }
  }
  __syncthreads();

  int bound[kRB];
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) {
    const int m = mc * kRowsC + 16 * rb + li;
    bound[rb] = m < M ? Lk - W + m % W : -1;
  }
  // Row 16 rb + li: the maximum (so far), and this lane's share of the sum
  // (kSum: the reciprocal of the row's sum).
  float m2[kRB], lsum[kRB];
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) {
    m2[rb] = kMode == kSum ? row_m[16 * rb + li] : -INFINITY;
    lsum[rb] = kMode == kSum ? row_r[16 * rb + li] : 0.f;
  }
  // The waves' shares of Y^T: columns 64 cg .. +63, keys kg * kpg .. of a step.
  const int CG = (D + 63) / 64, KG = kPartWaves / CG, kpg = kPartKeys / KG;
  const int cg = wv % CG, kg = wv / CG;
  f32x4 yacc[4][kRB];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) yacc[c][rb] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int t0 = 0; t0 < nrel; t0 += kPartKeys) {
    const int tw = t0 + 32 * wv;  // this wave's keys of the step
    f32x4 s[2][kRB];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) s[kb][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (tw < nrel) {
      const uint32_t r0 = (uint32_t)(tw + li) * kvs.k_rb, r1 = r0 + 16u * kvs.k_rb;
      for (int c0 = 0; c0 < nch; c0 += kGrp) {
        u32x4 k0[kGrp], k1[kGrp];
#pragma unroll
        for (int u = 0; u < kGrp; ++u) {
          const int col = (c0 + u) * kCols<T> + kEpl<T> * lg;
          const uint32_t cb = col * (uint32_t)sizeof(T);
          k0[u] = buf_load16(krs, col < D ? r0 + cb : kPastAll);
          k1[u] = buf_load16(krs, col < D ? r1 + cb : kPastAll);
        }
#pragma unroll
        for (int u = 0; u < kGrp; ++u)
          if (c0 + u < nch)
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
              const u32x4 qf = qop[(rb * nch + c0 + u) * 64 + lane];
              s[0][rb] = mfma_chunk<T>(k0[u], qf, s[0][rb]);
              s[1][rb] = mfma_chunk<T>(k1[u], qf, s[1][rb]);
            }
      }
    }
    float tm[kRB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      tm[rb] = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = tw + 16 * kb + 4 * lg + r;
          const float x = j < nrel && k_begin + j <= bound[rb] ? s[kb][rb][r] : -INFINITY;
          s[kb][rb][r] = x;
          tm[rb] = fmaxf(tm[rb], x);
        }
      if (kMode != kSum) tm[rb] = max_xor32(max_xor16(tm[rb]));
    }
    if constexpr (kMode == kStats) {
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        const float mn = fmaxf(m2[rb], tm[rb]), ms = mn == -INFINITY ? 0.f : mn;
        float ps = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) ps += __builtin_amdgcn_exp2f((s[kb][rb][r] - ms) * scale_log2);
        lsum[rb] = lsum[rb] * __builtin_amdgcn_exp2f((m2[rb] - ms) * scale_log2) + ps;
        m2[rb] = mn;
      }
    } else {
      if constexpr (kMode == kFlash) {
        // The step's row maxima over the workgroup.
        if (lg == 0)
#pragma unroll
          for (int rb = 0; rb < kRB; ++rb) wred[0][wv][16 * rb + li] = tm[rb];
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
          float mn = m2[rb];
#pragma unroll
          for (int w = 0; w < kPartWaves; ++w) mn = fmaxf(mn, wred[0][w][16 * rb + li]);
          const float ms = mn == -INFINITY ? 0.f : mn;
          const float alpha = __builtin_amdgcn_exp2f((m2[rb] - ms) * scale_log2);  // (0 at the first step)
          lsum[rb] *= alpha;
#pragma unroll
          for (int c = 0; c < 4; ++c) yacc[c][rb] *= alpha;
          m2[rb] = mn;
        }
      }
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        const float ms = m2[rb] == -INFINITY ? 0.f : m2[rb];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          f32x4 p;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[r] = __builtin_amdgcn_exp2f((s[kb][rb][r] - ms) * scale_log2);
            if (kMode == kSum)
              p[r] = s[kb][rb][r] == -INFINITY ? 0.f : round_through<T>(fminf(p[r] * lsum[rb], 1.f));
            else
              lsum[rb] += p[r];
          }
          *reinterpret_cast<f32x4*>(P + (16 * rb + li) * kPPitch + 32 * wv + 16 * kb + 4 * lg) = p;
        }
      }
      __syncthreads();
      if (kg < KG) {
        const uint32_t col = 64 * cg + 4 * li;
        const uint32_t cb = col * (uint32_t)sizeof(T);
        const int n = min(kpg, nrel - t0 - kg * kpg);
        for (int kk = 0; kk < n; kk += 32) {
          f32x4 v[2][4];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[h][e] = load4<T>(vrs, col < (uint32_t)D
                                          ? (uint32_t)(t0 + kg * kpg + kk + 16 * h + 4 * lg + e) * kvs.v_rb + cb
                                          : kPastAll);
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
              const f32x4 p = *reinterpret_cast<const f32x4*>(P + (16 * rb + li) * kPPitch + kg * kpg + kk + 16 * h +
                                                              4 * lg);
#pragma unroll
              for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < 4; ++c) yacc[c][rb] = mfma_f32(v[h][e][c], p[e], yacc[c][rb]);
            }
        }
      }
      __syncthreads();  // P and wred are rewritten by the next step
    }
  }

  if constexpr (kMode != kSum) {
    // Maxima and sums of the waves (kFlash: one maximum, shared).
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const float l = add_xor32(add_xor16(lsum[rb]));
      if (lg == 0) {
        wred[0][wv][16 * rb + li] = m2[rb];
        wred[1][wv][16 * rb + li] = l;
      }
    }
    __syncthreads();
    if (tid < R) {
      float mx = -INFINITY, l = 0.f;
      for (int w = 0; w < kPartWaves; ++w) mx = fmaxf(mx, wred[0][w][tid]);
      for (int w = 0; w < kPartWaves; ++w)
        if (wred[0][w][tid] != -INFINITY) l += wred[1][w][tid] * exp2f((wred[0][w][tid] - mx) * scale_log2);
      part_ml[(slot * kRowsC + tid) * 2] = mx;
      part_ml[(slot * kRowsC + tid) * 2 + 1] = l;
    }
  }
  if constexpr (kMode != kStats) {
    // Y of the KG key groups, added in order (over the operands and P, dead
    // since the last step's barrier).
    float* yb = reinterpret_cast<float*>(gm_lds);
    const int pitch = 64 * CG;
    if (kg < KG)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<f32x4*>(yb + (kg * R + 16 * rb + li) * pitch + 64 * cg + 16 * lg + 4 * r) =
              f32x4{yacc[0][rb][r], yacc[1][rb][r], yacc[2][rb][r], yacc[3][rb][r]};
    __syncthreads();
    const int d4 = D / 4;
    for (int i = tid; i < R * d4; i += NT) {
      const int row = i / d4, d = 4 * (i % d4);
      f32x4 y = *reinterpret_cast<const f32x4*>(yb + row * pitch + d);
      for (int k = 1; k < KG; ++k) y += *reinterpret_cast<const f32x4*>(yb + (k * R + row) * pitch + d);
      *reinterpret_cast<f32x4*>(part_y + (slot * kRowsC + row) * D + d) = y;
    }
  }
}

// ---------------------------------------------------------------------------
// One wave per (head, query row): the log-sum-exp over the splits and y, four
// columns a lane.  flash: the partials are relative to their split's maximum.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(64)
genm_merge_kernel(const float* __restrict__ part_ml, const float* __restrict__ part_y, int n_mc, int n_splits, int M,
                  int D, float scale_log2, int flash, int y_round, float* __restrict__ ystat, float* __restrict__ yf32,
                  float* __restrict__ row_mr, uint32_t* __restrict__ zero_ptr, int64_t zero_words) {
  const int lane = threadIdx.x, head = blockIdx.x / M, m = blockIdx.x % M;
  const int mc = m / kRowsC, row = m % kRowsC;
  const int64_t slot0 = ((int64_t)head * n_mc + mc) * n_splits;
  const float* ml = part_ml + (slot0 * kRowsC + row) * 2;
  const bool col = 4 * lane < D;
  const float* py = part_y + (slot0 * kRowsC + row) * D + (col ? 4 * lane : 0);
  float mx = -INFINITY;
  for (int s = lane; s < n_splits; s += 64) mx = fmaxf(mx, ml[s * kRowsC * 2]);
  mx = wave_max_dpp(mx);
  float l = 0.f;
  for (int s = lane; s < n_splits; s += 64) {
    const float ms = ml[s * kRowsC * 2];
    if (ms != -INFINITY) l += ml[s * kRowsC * 2 + 1] * exp2f((ms - mx) * scale_log2);
  }
  l = wave_sum_dpp(l);
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < n_splits; ++s) {
    const f32x4 ys = *reinterpret_cast<const f32x4*>(py + (int64_t)s * kRowsC * D);
    const float ms = ml[s * kRowsC * 2];
    const float f = !flash ? 1.f : ms == -INFINITY ? 0.f : exp2f((ms - mx) * scale_log2);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = fmaf(f, ys[e], y[e]);
  }
  const int mpad = n_mc * kRowsC;
  const int64_t rbase = (int64_t)head * mpad + m;
  float yy = 0.f;
  const float rl = 1.f / l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (flash) y[e] *= rl;
    if (y_round) y[e] = round_through<T>(y[e]);
    yy = fmaf(y[e], y[e], yy);
  }
  if (col) *reinterpret_cast<f32x4*>(yf32 + rbase * D + 4 * lane) = y;
  yy = wave_sum_dpp(col ? yy : 0.f);
  if (lane == 0) {
    ystat[rbase * 2 + 0] = mx * scale_log2 + log2f(l);
    ystat[rbase * 2 + 1] = yy;
    if (flash) reinterpret_cast<float2*>(row_mr)[rbase] = make_float2(mx, rl);  // (else part<kSum> wrote them)
  }
  if (zero_ptr)
    for (int64_t i = (int64_t)blockIdx.x * 64 + lane; i < zero_words; i += (int64_t)gridDim.x * 64) zero_ptr[i] = 0u;
}

// ---------------------------------------------------------------------------
// Scores.  One workgroup per (head, kpw keys); a wave takes 16 keys at a time:
// S = Q K^T and G = Y V^T with rows on the result registers and keys on the
// lanes, so that a key's sum over the rows is in-lane but for the four lane
// groups.  Q and Y of 16 * kRB rows at a time in LDS in operand order; the
// keys' sums over earlier rows in LDS.  kYT: Y was rounded to T, so T operands
// hold it exactly.
// ---------------------------------------------------------------------------
template <typename T, int kRB, bool kYT>
__global__ void __launch_bounds__(64 * kScoreWaves)
genm_score_kernel(const T* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_sd,
                  const T* __restrict__ kp, const T* __restrict__ vp, KvStride kvs, int Hkv, int Lq, int Lk, int D,
                  int W, int g, int M, int mpad, float scale_log2, float eps, int p_round, int wgs, int kpw,
                  const float* __restrict__ ystat, const float* __restrict__ yf32, const float* __restrict__ row_mr,
                  float* __restrict__ scores) {
  constexpr int NT = 64 * kScoreWaves;
  constexpr int R = 16 * kRB;
  constexpr int YV = kYT ? 1 : kEpl<T> / 4;  // 16-byte units of Y per lane and chunk
  extern __shared__ u32x4 gm_lds[];
  __shared__ __attribute__((aligned(16))) float row_m[kRowsC], row_r[kRowsC];
  __shared__ __attribute__((aligned(16))) float yn2[kRowsC];
  const int nch = (D + kCols<T> - 1) / kCols<T>;
  u32x4* qop = gm_lds;
  u32x4* yop = qop + kRB * nch * 64;                          // [kRB][nch][YV][64]
  float* sc = reinterpret_cast<float*>(yop + kRB * nch * YV * 64);  // [kpw]

  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int head = lid / wgs, k_begin = (lid % wgs) * kpw, nrel = min(kpw, Lk - k_begin);
  const int b = head / Hkv, hkv = head % Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lg = lane >> 4;
  const rsrc_t krs = make_rsrc(reinterpret_cast<const char*>(kp + b * kvs.k_sb + hkv * kvs.k_sh) +
                                   (int64_t)k_begin * kvs.k_rb,
                               rows_bytes(nrel, kvs.k_rb, D * (uint32_t)sizeof(T)));
  const char* vhead = reinterpret_cast<const char*>(vp + b * kvs.v_sb + hkv * kvs.v_sh) + (int64_t)k_begin * kvs.v_rb;
  const rsrc_t vrs = make_rsrc(vhead, rows_bytes(nrel, kvs.v_rb, D * (uint32_t)sizeof(T)));
  const float inv_g = static_cast<float>(g);

  for (int r0 = 0; r0 < M; r0 += R) {
    if (r0) __syncthreads();  // the previous rows' operands are dead
    stage_q<T, kRB, NT>(qop, nch, q, q_sb, q_sh, q_ss, q_sd, b, hkv, g, W, Lq, M, D, r0);
    const float* yrow0 = yf32 + ((int64_t)head * mpad + r0) * D;
    for (int s = tid; s < kRB * nch * 64; s += NT) {
      const int l = s & 63, c = (s >> 6) % nch, rb = (s >> 6) / nch;
      const int row = 16 * rb + (l & 15), d0 = c * kCols<T> + kEpl<T> * (l >> 4);
      const bool in = r0 + row < M && d0 < D;  // (D is a multiple of kEpl)
      float y[kEpl<T>];
#pragma unroll
      for (int e = 0; e < kEpl<T>; ++e) y[e] = in ? yrow0[(int64_t)row * D + d0 + e] : 0.f;
      if constexpr (kYT) {
        T x[kEpl<T>];
#pragma unroll
        for (int e = 0; e < kEpl<T>; ++e) x[e] = static_cast<T>(y[e]);
        u32x4 w;
        __builtin_memcpy(&w, x, 16);
        yop[s] = w;
      } else {
#pragma unroll
        for (int u = 0; u < YV; ++u) {
          u32x4 w;
          __builtin_memcpy(&w, y + 4 * u, 16);
          yop[((rb * nch + c) * YV + u) * 64 + l] = w;
        }
      }
    }
    if (tid < R) {
      const bool in = r0 + tid < M;
      const int64_t i = ((int64_t)head * mpad + r0 + tid) * 2;
      row_m[tid] = in ? row_mr[i] : 0.f;
      row_r[tid] = in ? row_mr[i + 1] : 0.f;
      yn2[tid] = in ? ystat[i + 1] : 0.f;
    }
    __syncthreads();
    int bound[kRB][4];
    f32x4 m4[kRB], r4[kRB], y4[kRB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      m4[rb] = *reinterpret_cast<const f32x4*>(row_m + 16 * rb + 4 * lg);
      r4[rb] = *reinterpret_cast<const f32x4*>(row_r + 16 * rb + 4 * lg);
      y4[rb] = *reinterpret_cast<const f32x4*>(yn2 + 16 * rb + 4 * lg);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = r0 + 16 * rb + 4 * lg + r;
        bound[rb][r] = m < M ? Lk - W + m % W - k_begin : -1;  // last visible key, relative to k_begin
      }
    }

    for (int t = 16 * wv; t < nrel; t += 16 * kScoreWaves) {
      f32x4 s[kRB], gg[kRB];
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) s[rb] = gg[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
      float vsq = 0.f;
      const uint32_t kr = (uint32_t)(t + li) * kvs.k_rb, vr = (uint32_t)(t + li) * kvs.v_rb;
      for (int c0 = 0; c0 < nch; c0 += kGrp) {
        u32x4 kf[kGrp], vf[kGrp];
#pragma unroll
        for (int u = 0; u < kGrp; ++u) {
          const int col = (c0 + u) * kCols<T> + kEpl<T> * lg;
          const uint32_t cb = col * (uint32_t)sizeof(T);
          kf[u] = buf_load16(krs, col < D ? kr + cb : kPastAll);
          vf[u] = buf_load16(vrs, col < D ? vr + cb : kPastAll);
        }
#pragma unroll
        for (int u = 0; u < kGrp; ++u)
          if (c0 + u < nch) {
            float ve[kEpl<T>];
#pragma unroll
            for (int e = 0; e < kEpl<T>; ++e) {
              ve[e] = elem_of<T>(vf[u], e);
              vsq = fmaf(ve[e], ve[e], vsq);
            }
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
              const int ch = rb * nch + c0 + u;
              s[rb] = mfma_chunk<T>(qop[ch * 64 + lane], kf[u], s[rb]);
              if constexpr (kYT) {
                gg[rb] = mfma_chunk<T>(yop[ch * 64 + lane], vf[u], gg[rb]);
              } else {
#pragma unroll
                for (int w = 0; w < YV; ++w) {
                  const f32x4 yf = __builtin_bit_cast(f32x4, yop[(ch * YV + w) * 64 + lane]);
#pragma unroll
                  for (int e = 0; e < 4; ++e) gg[rb] = mfma_f32(yf[e], ve[4 * w + e], gg[rb]);
                }
              }
            }
          }
      }
      const float vn2 = add_xor32(add_xor16(vsq));
      float sum = 0.f;
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool seen = t + li <= bound[rb][r] && t + li < nrel;
          float p = fminf(__builtin_amdgcn_exp2f((s[rb][r] - m4[rb][r]) * scale_log2) * r4[rb][r], 1.f);
          if (p_round) p = round_through<T>(p);
          const float terms = vn2 + y4[rb][r];
          float d2 = fmaf(-2.f, gg[rb][r], terms);
          // (NaN counts as cancelled, so that infinite rows give what the
          // direct form gives.)
          uint64_t need = __ballot(seen && !(d2 >= kDirect * terms));
          while (need) {
            const int l = __builtin_ctzll(need);
            need &= need - 1;
            const int key = t + (l & 15), row = 16 * rb + 4 * (l >> 4) + r;
            const T* vrow = reinterpret_cast<const T*>(vhead + (int64_t)key * kvs.v_rb);
            const float* yrow = yrow0 + (int64_t)row * D;
            float a = 0.f;
            for (int d = lane; d < D; d += 64) {
              const float x = static_cast<float>(vrow[d]) - yrow[d];
              a = fmaf(x, x, a);
            }
            a = wave_sum_dpp(a);
            d2 = lane == l ? a : d2;
          }
          const float ratio = p / (1.f - p + eps);
          sum = seen ? fmaf(ratio * ratio, d2, sum) : sum;
        }
      sum = add_xor16(add_xor32(sum));
      if (lg == 0) {
        if (r0) sum += sc[t + li];
        if (r0 + R >= M) {
          if (t + li < nrel) scores[(int64_t)head * Lk + k_begin + t + li] = sum / inv_g;
        } else {
          sc[t + li] = sum;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
template <typename T, int kRB>
static hipError_t launch_genm_t(const ScorePlan& p, int D, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                                int64_t q_sd, const KvSrc& kv, int Hkv, int Lq, int Lk, int W, float eps, int p_round,
                                int y_round, float* scores, char* ws, uint32_t* zero_ptr, int64_t zero_words,
                                hipStream_t st) {
  const float scale_log2 = 1.4426950408889634f / sqrtf((float)D);
  float* part_ml = reinterpret_cast<float*>(ws + p.off_ml);
  float* part_y = reinterpret_cast<float*>(ws + p.off_y);
  float* ystat = reinterpret_cast<float*>(ws + p.off_stat);
  float* yf = reinterpret_cast<float*>(ws + p.off_yf);
  // (maximum, 1 / sum) per row: 2 of the kMB * kStatWords / 32 = 4 words per
  // row that the plan holds for pass 2's statistics, unused here.
  float* row_mr = reinterpret_cast<float*>(ws + p.off_stb);
  const T* qq = static_cast<const T*>(q);
  const T* kk = static_cast<const T*>(kv.k);
  const T* vv = static_cast<const T*>(kv.v);
  const KvStride kvs = kv_strides(kv, sizeof(T));
  const bool flash = sizeof(T) == 4 || !p_round;  // fp32: rounding p is the identity
  const int nch = (D + kCols<T> - 1) / kCols<T>;
  const int CG = (D + 63) / 64, KG = kPartWaves / CG;
  const size_t ops = (size_t)kRB * nch * 64 * 16;
  const size_t lds1 = std::max(ops + (size_t)16 * kRB * kPPitch * 4, (size_t)KG * 16 * kRB * CG * 64 * 4);
  const dim3 g1(p.heads * p.n_mc * p.s1), b1(64 * kPartWaves);
  auto part = [&](auto kern, size_t lds) {
    launch(kern, g1, b1, lds, st, qq, q_sb, q_sh, q_ss, q_sd, kk, vv, kvs, Hkv, Lq, Lk, D, W, p.g, p.M, p.n_mc, p.s1,
           p.kps1, scale_log2, part_ml, part_y, row_mr);
  };
  if (flash) {
    part(genm_part_kernel<T, kRB, kFlash>, lds1);
  } else {
    part(genm_part_kernel<T, kRB, kStats>, ops);
    part(genm_part_kernel<T, kRB, kSum>, lds1);
  }
  launch(genm_merge_kernel<T>, dim3(p.heads * p.M), dim3(64), 0, st, part_ml, part_y, p.n_mc, p.s1, p.M, D,
         scale_log2, flash ? 1 : 0, y_round, ystat, yf, row_mr, zero_ptr, zero_words);
  // Keys per workgroup: 64 (16 per wave) until there are more workgroups than
  // the GPU runs at once, then more, so that staging Q and Y is shared.
  constexpr int kStep = 16 * kScoreWaves;
  const int steps = (Lk + kStep - 1) / kStep;
  const int per = std::min(16, std::max(1, (int)(((int64_t)p.heads * steps + 1023) / 1024)));
  const int kpw = per * kStep, wgs = (Lk + kpw - 1) / kpw;
  auto score = [&](auto kern, size_t yv) {
    launch(kern, dim3(p.heads * wgs), dim3(64 * kScoreWaves), ops * (1 + yv) + (size_t)kpw * 4, st, qq, q_sb, q_sh,
           q_ss, q_sd, kk, vv, kvs, Hkv, Lq, Lk, D, W, p.g, p.M, p.mpad, scale_log2, eps, p_round, wgs, kpw, ystat,
           yf, row_mr, scores);
  };
  if constexpr (sizeof(T) == 2) {
    if (y_round)
      score(genm_score_kernel<T, kRB, true>, 1);
    else
      score(genm_score_kernel<T, kRB, false>, 2);
  } else {
    score(genm_score_kernel<T, kRB, false>, 1);
  }
  return hipGetLastError();
}

bool generic_on_mfma(int dtype, int64_t D, int64_t Lk, const KvSrc& kv) {
  const int64_t eb = dtype == kDtypeFp32 ? 4 : 2;
  // Rows of whole 16-byte units (the operand loads), up to the 256 columns
  // whose sums the part kernel's eight waves hold, within 32-bit offsets.
  return D <= 256 && (D * eb) % 16 == 0 && kv_rows_fit(kv.k_sl, eb, Lk, D) && kv_rows_fit(kv.v_sl, eb, Lk, D);
}

hipError_t launch_scores_generic_mfma(const ScorePlan& p, int dtype, int D, const void* q, int64_t q_sb, int64_t q_sh,
                                      int64_t q_ss, int64_t q_sd, const KvSrc& kv, int Hkv, int Lq, int Lk, int W,
                                      float eps, int p_round, int y_round, float* scores, char* ws,
                                      uint32_t* zero_ptr, int64_t zero_words, hipStream_t st) {
#define DKV_CASE(TT)                                                                                              \
  return p.M <= 16 ? launch_genm_t<TT, 1>(p, D, q, q_sb, q_sh, q_ss, q_sd, kv, Hkv, Lq, Lk, W, eps, p_round, y_round, \
                                          scores, ws, zero_ptr, zero_words, st)                                   \
                   : launch_genm_t<TT, 2>(p, D, q, q_sb, q_sh, q_ss, q_sd, kv, Hkv, Lq, Lk, W, eps, p_round, y_round, \
                                          scores, ws, zero_ptr, zero_words, st)
  if (dtype == kDtypeBf16) DKV_CASE(__bf16);
  if (dtype == kDtypeFp16) DKV_CASE(_Float16);
  DKV_CASE(float);
#undef DKV_CASE
}

}  // namespace dkv
