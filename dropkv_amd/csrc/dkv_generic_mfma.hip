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
// Values that are not finite: y is a sum over all keys of a tile, with p = 0 for
// the keys a row does not see, so that an infinite or NaN value in the last W
// keys makes y NaN for the rows before it too (0 * inf; so do p @ V in torch and
// pass 1 of the tuned pipeline).  The vector-ALU kernels stop at each row's last
// key.  No finite score is lost by it: the last row sees every key, and its y is
// not finite either way.
//
// What bounds them: at the sizes these inputs are used at (a few thousand
// keys), latency: three or four launches, and in each one round trip to memory
// for the operands, the matrix instructions of a tile and a reduction.  The
// vector-ALU kernels read K with one row per lane (16 lanes of a load in 16
// different rows) and gave each query row a workgroup of its own: 3990 us for
// 8192 keys of D 256 in bf16 (8 query, 4 KV heads), 3650 us for 8192 keys of D
// 64 in fp32 (14, 2), 1790 us for 4099 keys of D 96 in fp16 (16, 16); these
// kernels take 37, 29 and 32 us.  With the operand loads issued one round trip
// after the other (a wait for a load waits for every earlier one, so the query
// rows go before K and V), Q and Y staged 32 rows at a time and y's columns 64
// words apart in LDS they took 49, 34 and 34 us.
//
// These are figures for values of zero mean.  Values that share a mean of more
// than about 1.2 times their spread have every distance taken directly, one (key,
// row) pair of a wave after the other: with a mean of 3 and a spread of 1 the
// same calls take 183, 207 and 103 us (the vector-ALU kernels, which take every
// distance directly, the same 3990, 3650 and 1790).  With many rows per KV head
// the two are closest: 32 query heads of D 256 on 2 KV heads, a window of 16 and
// 2100 keys take 2.1 ms, and 5.8 ms there.
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

// Groups of waves that share a step's keys when CG of them share the columns.
__host__ __device__ constexpr int part_kg(int CG) { return CG == 1 ? 8 : CG == 2 ? 4 : 2; }

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

// Where query row m of the group starts (rows past M: the last one).
template <typename T>
__device__ __forceinline__ const T* q_row(const T* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_ss, int b,
                                          int hkv, int g, const Div& dw, int Lq, int M, int m) {
  const int mm = min(m, M - 1), gi = dw.div(mm);
  return q + (int64_t)b * q_sb + (int64_t)(hkv * g + gi) * q_sh + (int64_t)(Lq - (int)dw.d + mm - gi * (int)dw.d) * q_ss;
}

// A lane's 16 bytes of an MFMA operand: kEpl elements of a row by stride.
template <typename T>
__device__ __forceinline__ u32x4 gather_unit(const T* row, int64_t sd) {
  T x[kEpl<T>];
#pragma unroll
  for (int e = 0; e < kEpl<T>; ++e) x[e] = row[(int64_t)e * sd];
  u32x4 w;
  __builtin_memcpy(&w, x, 16);
  return w;
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
genm_part_kernel(const T* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_sd, bool qvec,
                 const T* __restrict__ kp, const T* __restrict__ vp, KvStride kvs, int Hkv, int Lq, int Lk, int D,
                 int W, int g, int M, int n_mc, int n_splits, int kps, float scale_log2,
                 float* __restrict__ part_ml, float* __restrict__ part_y, float* __restrict__ row_mr,
                 ScoreDiv dv) {
  constexpr int R = 16 * kRB;
  extern __shared__ u32x4 gm_lds[];
  __shared__ float wred[2][kPartWaves][kRowsC];
  __shared__ float row_m[kRowsC], row_r[kRowsC];  // kSum: the rows' maxima and 1 / sums
  const int nch = (D + kCols<T> - 1) / kCols<T>;
  u32x4* qop = gm_lds;
  float* P = reinterpret_cast<float*>(qop + kRB * nch * 64);

  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int mc = dv.n_mc.mod(lid), hs = dv.n_mc.div(lid);
  const int split = dv.splits.mod(hs), head = dv.splits.div(hs);
  const int b = dv.hkv.div(head), hkv = dv.hkv.mod(head);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int k_begin = split * kps, k_end = min(k_begin + kps, Lk), nrel = k_end - k_begin;
  const rsrc_t krs = make_rsrc(reinterpret_cast<const char*>(kp + b * kvs.k_sb + hkv * kvs.k_sh) +
                                   (int64_t)k_begin * kvs.k_rb,
                               rows_bytes(nrel, kvs.k_rb, D * (uint32_t)sizeof(T)));
  const rsrc_t vrs = make_rsrc(reinterpret_cast<const char*>(vp + b * kvs.v_sb + hkv * kvs.v_sh) +
                                   (int64_t)k_begin * kvs.v_rb,
                               rows_bytes(nrel, kvs.v_rb, D * (uint32_t)sizeof(T)));
  const int64_t slot = ((int64_t)head * n_mc + mc) * n_splits + split;

  // Loads of the wave's 32 keys at t, chunks c0 .. c0 + kGrp - 1, and of 32 keys
  // of its share of V from row t of a step; the first of both are on their way
  // while the operands are staged.
  u32x4 k0[kGrp], k1[kGrp];
  auto load_k = [&](int t, int c0) __attribute__((always_inline)) {
    const uint32_t r0 = (uint32_t)(t + li) * kvs.k_rb, r1 = r0 + 16u * kvs.k_rb;
#pragma unroll
    for (int u = 0; u < kGrp; ++u) {
      const int col = (c0 + u) * kCols<T> + kEpl<T> * lg;
      const uint32_t cb = col * (uint32_t)sizeof(T);
      k0[u] = buf_load16(krs, col < D ? r0 + cb : kPastAll);
      k1[u] = buf_load16(krs, col < D ? r1 + cb : kPastAll);
    }
  };
  const int CG = (D + 63) / 64, KG = part_kg(CG), kpg = kPartKeys / kPartWaves * (CG == 3 ? 4 : CG);
  const int kg = CG == 3 ? (wv * 11) >> 5 : wv >> (CG / 2), cg = wv - kg * CG;  // wv / CG, wv % CG
  const uint32_t v_col = 64 * cg + 4 * li;
  auto load_v = [&](f32x4 (&v)[2][4], int t) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[h][e] = load4<T>(vrs, v_col < (uint32_t)D && kg < KG
                                    ? (uint32_t)(t + 16 * h + 4 * lg + e) * kvs.v_rb + v_col * (uint32_t)sizeof(T)
                                    : kPastAll);
  };
  f32x4 va[2][4], vb[2][4];
  // A wait for a load also waits for every load issued before it: the query
  // rows (and the splits' statistics) first, then K and V.  Slot (rb, chunk,
  // lane) of qop holds the lane's 16 bytes; wave w takes chunks w and w + 8.
  static_assert(2 * kPartWaves * kCols<float> >= 256, "two chunks a wave");
  u32x4 qr[kRB][2];
  const T* qrow[kRB];
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb)
    qrow[rb] = q_row(q, q_sb, q_sh, q_ss, b, hkv, g, dv.w, Lq, M, mc * kRowsC + 16 * rb + li);
  const int qd = wv * kCols<T> + kEpl<T> * lg;  // column of the wave's first chunk
  if (qvec)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int d0 = qd + i * kPartWaves * kCols<T>;
        qr[rb][i] = *reinterpret_cast<const u32x4*>(qrow[rb] + (d0 < D ? d0 : 0));
      }
  constexpr int kMl = 4;  // splits per thread read up front (16 threads a row)
  f32x2 mlv[kMl];
  const rsrc_t mrs = make_rsrc(part_ml + ((int64_t)head * n_mc + mc) * n_splits * kRowsC * 2,
                               (uint32_t)n_splits * kRowsC * 8u);
  const int srow = tid >> 4;  // the row whose statistics this thread helps to combine
  if constexpr (kMode == kSum)
#pragma unroll
    for (int i = 0; i < kMl; ++i) mlv[i] = buf_load8f(mrs, ((uint32_t)((tid & 15) + 16 * i) * kRowsC + srow) * 8u);
  load_k(32 * wv, 0);
  if constexpr (kMode != kStats) load_v(va, kg * kpg);
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (wv + kPartWaves * i < nch) {
        const int d0 = qd + i * kPartWaves * kCols<T>;
        if (!qvec) qr[rb][i] = gather_unit(qrow[rb] + (int64_t)(d0 < D ? d0 : 0) * q_sd, q_sd);
        qop[(rb * nch + wv + kPartWaves * i) * 64 + lane] =
            mc * kRowsC + 16 * rb + li < M && d0 < D ? qr[rb][i] : u32x4{0u, 0u, 0u, 0u};
      }
  if constexpr (kMode == kSum) {
    // The rows' maxima and sums from the splits': 16 threads a row.
    const int row = srow, s0 = tid & 15;
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < kMl; ++i) mx = s0 + 16 * i < n_splits ? fmaxf(mx, mlv[i][0]) : mx;
    for (int s = s0 + 16 * kMl; s < n_splits; s += 16)
      mx = fmaxf(mx, buf_load8f(mrs, ((uint32_t)s * kRowsC + row) * 8u)[0]);
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    float l = 0.f;
    auto part = [&](f32x2 p) { return p[0] == -INFINITY ? 0.f : p[1] * exp2f((p[0] - mx) * scale_log2); };
#pragma unroll
    for (int i = 0; i < kMl; ++i) l += s0 + 16 * i < n_splits ? part(mlv[i]) : 0.f;
    for (int s = s0 + 16 * kMl; s < n_splits; s += 16) l += part(buf_load8f(mrs, ((uint32_t)s * kRowsC + row) * 8u));
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
    bound[rb] = m < M ? Lk - W + dv.w.mod(m) : -1;
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
    for (int c0 = 0; c0 < nch; c0 += kGrp) {
      if (c0) load_k(tw, c0);
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
    if (t0 + kPartKeys < nrel) load_k(tw + kPartKeys, 0);
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
        // 32 keys at a time, the next 32 on their way (the last ones of a step:
        // the next step's first).
        const int n = min(kpg, nrel - t0 - kg * kpg);
        auto add = [&](const f32x4 (&v)[2][4], int kk) __attribute__((always_inline)) {
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
        };
        const int next = t0 + kPartKeys + kg * kpg;
        for (int kk = 0; kk < kpg; kk += 64) {
          const int r = t0 + kg * kpg + kk;
          load_v(vb, kk + 32 < kpg ? r + 32 : next);
          if (kk < n) add(va, kk);
          if (kk + 32 < kpg) {
            load_v(va, kk + 64 < kpg ? r + 64 : next);
            if (kk + 32 < n) add(vb, kk + 32);
          } else {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int e = 0; e < 4; ++e) va[h][e] = vb[h][e];
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
    const int pitch = 64 * CG + 4;  // (rows of 64 words would share their banks)
    if (kg < KG)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<f32x4*>(yb + (kg * R + 16 * rb + li) * pitch + 64 * cg + 16 * lg + 4 * r) =
              f32x4{yacc[0][rb][r], yacc[1][rb][r], yacc[2][rb][r], yacc[3][rb][r]};
    __syncthreads();
    const int d = 4 * lane;
    for (int row = wv; row < R && d < D; row += kPartWaves) {
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
  const int lane = threadIdx.x, head = blockIdx.y, m = blockIdx.x;
  const int mc = m / kRowsC, row = m % kRowsC;
  const int64_t slot0 = ((int64_t)head * n_mc + mc) * n_splits;
  const float* ml = part_ml + (slot0 * kRowsC + row) * 2;
  const bool col = 4 * lane < D;
  float mx = -INFINITY;
  for (int s = lane; s < n_splits; s += 64) mx = fmaxf(mx, ml[s * kRowsC * 2]);
  mx = wave_max_dpp(mx);
  float l = 0.f;
  for (int s = lane; s < n_splits; s += 64) {
    const float ms = ml[s * kRowsC * 2];
    if (ms != -INFINITY) l += ml[s * kRowsC * 2 + 1] * exp2f((ms - mx) * scale_log2);
  }
  l = wave_sum_dpp(l);
  // y in batches of 32 splits whose loads are all issued together (zeros past
  // the last split and past column D).
  const rsrc_t yrs = make_rsrc(part_y + slot0 * kRowsC * D, (uint32_t)n_splits * kRowsC * D * 4u);
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < n_splits; s0 += 32) {
    f32x4 ys[32];
#pragma unroll
    for (int u = 0; u < 32; ++u)
      ys[u] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     yrs, 4 * lane < D && s0 + u < n_splits ? (((uint32_t)(s0 + u) * kRowsC + row) * D + 4 * lane) * 4u
                                                            : kPastAll, 0, 0));
    const float ms = s0 + (lane & 31) < n_splits ? ml[(s0 + (lane & 31)) * kRowsC * 2] : -INFINITY;
    const float fl = !flash ? 1.f : ms == -INFINITY ? 0.f : exp2f((ms - mx) * scale_log2);
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      const float f = read_lane_f(fl, u);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fmaf(f, ys[u][e], y[e]);
    }
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
    for (int64_t i = ((int64_t)head * M + m) * 64 + lane; i < zero_words; i += (int64_t)gridDim.x * gridDim.y * 64)
      zero_ptr[i] = 0u;
}

// ---------------------------------------------------------------------------
// Scores.  One workgroup per (head, kpw keys); a wave takes 16 keys at a time:
// S = Q K^T and G = Y V^T with rows on the result registers and keys on the
// lanes, so that a key's sum over the rows is in-lane but for the four lane
// groups.  Q and Y of `rs` rows at a time (all of them where LDS allows) in
// operand order; a tile's K and V stay in registers for all of them (up to
// eight chunks); the keys' sums over earlier rows in LDS.  kYT: Y was rounded
// to T, so T operands hold it exactly.
// ---------------------------------------------------------------------------
template <typename T, int kRB, bool kYT>
__global__ void __launch_bounds__(64 * kScoreWaves)
genm_score_kernel(const T* __restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_sd, bool qvec,
                  const T* __restrict__ kp, const T* __restrict__ vp, KvStride kvs, int Hkv, int Lq, int Lk, int D,
                  int W, int g, int M, int mpad, float scale_log2, float eps, int p_round, int kpw, int rs,
                  const float* __restrict__ ystat, const float* __restrict__ yf32, const float* __restrict__ row_mr,
                  float* __restrict__ scores, ScoreDiv dv) {
  constexpr int NT = 64 * kScoreWaves;
  constexpr int R = 16 * kRB;
  constexpr int YV = kYT ? 1 : kEpl<T> / 4;  // 16-byte units of Y per lane and chunk
  extern __shared__ u32x4 gm_lds[];
  const int nch = (D + kCols<T> - 1) / kCols<T>;
  u32x4* qop = gm_lds;                                        // [rs / 16][nch][64]
  u32x4* yop = qop + rs / 16 * nch * 64;                      // [rs / 16][nch][YV][64]
  f32x4* st = reinterpret_cast<f32x4*>(yop + rs / 16 * nch * YV * 64);  // [rs / 16][3][4]: maxima, 1 / sums, |y|^2
  float* stf = reinterpret_cast<float*>(st);
  float* sc = stf + rs * 3;                                   // [kpw]

  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int head = dv.splits.div(lid), k_begin = dv.splits.mod(lid) * kpw, nrel = min(kpw, Lk - k_begin);
  const int b = dv.hkv.div(head), hkv = dv.hkv.mod(head);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lg = lane >> 4;
  const rsrc_t krs = make_rsrc(reinterpret_cast<const char*>(kp + b * kvs.k_sb + hkv * kvs.k_sh) +
                                   (int64_t)k_begin * kvs.k_rb,
                               rows_bytes(nrel, kvs.k_rb, D * (uint32_t)sizeof(T)));
  const char* vhead = reinterpret_cast<const char*>(vp + b * kvs.v_sb + hkv * kvs.v_sh) + (int64_t)k_begin * kvs.v_rb;
  const rsrc_t vrs = make_rsrc(vhead, rows_bytes(nrel, kvs.v_rb, D * (uint32_t)sizeof(T)));

  u32x4 kf[kGrp], vf[kGrp];
  auto load = [&](int t, int c0) __attribute__((always_inline)) {
    const uint32_t kr = (uint32_t)(t + li) * kvs.k_rb, vr = (uint32_t)(t + li) * kvs.v_rb;
#pragma unroll
    for (int u = 0; u < kGrp; ++u) {
      const int col = (c0 + u) * kCols<T> + kEpl<T> * lg;
      const uint32_t cb = col * (uint32_t)sizeof(T);
      kf[u] = buf_load16(krs, col < D ? kr + cb : kPastAll);
      vf[u] = buf_load16(vrs, col < D ? vr + cb : kPastAll);
    }
  };
  const bool once = nch <= kGrp;  // a tile's K and V fit the registers

  for (int r0 = 0; r0 < M; r0 += rs) {
    if (r0) __syncthreads();  // the previous rows' operands are dead
    const int nrb = min(rs, (M - r0 + R - 1) / R * R) / 16;
    const float* yrow0 = yf32 + ((int64_t)head * mpad + r0) * D;
    // Q and Y, kRB row blocks and eight chunks at a time (wave w takes chunks w
    // and w + 4), every load of a batch issued before its first LDS write, and
    // the first tile's K and V behind the first batch's.
    constexpr int YU = kEpl<T> / 4;
    for (int rb0 = 0; rb0 < nrb; rb0 += kRB)
      for (int c0 = 0; c0 < nch; c0 += 2 * kScoreWaves) {
        u32x4 qr[kRB][2];
        f32x4 yr[kRB][2][YU];
        const T* qrow[kRB];
        const int qd = (c0 + wv) * kCols<T> + kEpl<T> * lg;
#pragma unroll
        for (int i = 0; i < kRB; ++i) {
          const int m = r0 + 16 * (rb0 + i) + li;
          qrow[i] = q_row(q, q_sb, q_sh, q_ss, b, hkv, g, dv.w, Lq, M, m);
          const float* yrow = yrow0 + (int64_t)(min(m, M - 1) - r0) * D;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int d0 = qd + j * kScoreWaves * kCols<T>, dc = d0 < D ? d0 : 0;
            if (qvec) qr[i][j] = *reinterpret_cast<const u32x4*>(qrow[i] + dc);
#pragma unroll
            for (int u = 0; u < YU; ++u) yr[i][j][u] = *reinterpret_cast<const f32x4*>(yrow + dc + 4 * u);
          }
        }
        if (r0 == 0 && rb0 == 0 && c0 == 0) load(16 * wv, 0);
#pragma unroll
        for (int i = 0; i < kRB; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int c = c0 + wv + kScoreWaves * j, ch = (rb0 + i) * nch + c, d0 = qd + j * kScoreWaves * kCols<T>;
            if (c < nch) {
              const bool in = r0 + 16 * (rb0 + i) + li < M && d0 < D;
              if (!qvec) qr[i][j] = gather_unit(qrow[i] + (int64_t)(d0 < D ? d0 : 0) * q_sd, q_sd);
              qop[ch * 64 + lane] = in ? qr[i][j] : u32x4{0u, 0u, 0u, 0u};
              f32x4 y[YU];
#pragma unroll
              for (int u = 0; u < YU; ++u) y[u] = in ? yr[i][j][u] : f32x4{0.f, 0.f, 0.f, 0.f};
              if constexpr (kYT) {
                T x[kEpl<T>];
#pragma unroll
                for (int e = 0; e < kEpl<T>; ++e) x[e] = static_cast<T>(y[e / 4][e % 4]);
                u32x4 w;
                __builtin_memcpy(&w, x, 16);
                yop[ch * 64 + lane] = w;
              } else {
#pragma unroll
                for (int u = 0; u < YU; ++u) yop[(ch * YV + u) * 64 + lane] = __builtin_bit_cast(u32x4, y[u]);
              }
            }
          }
      }
    for (int r = tid; r < 16 * nrb; r += NT) {
      const bool in = r0 + r < M;
      const int64_t i = ((int64_t)head * mpad + (in ? r0 + r : 0)) * 2;
      stf[(r / 16 * 3 + 0) * 16 + r % 16] = in ? row_mr[i] : 0.f;
      stf[(r / 16 * 3 + 1) * 16 + r % 16] = in ? row_mr[i + 1] : 0.f;
      stf[(r / 16 * 3 + 2) * 16 + r % 16] = in ? ystat[i + 1] : 0.f;
    }
    __syncthreads();

    for (int t = 16 * wv; t < nrel; t += 16 * kScoreWaves) {
      if (once && (r0 || t != 16 * wv)) load(t, 0);
      float total = 0.f, vn2 = 0.f;
      for (int g0 = 0; g0 < nrb; g0 += kRB) {
        f32x4 s[kRB], gg[kRB];
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) s[rb] = gg[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
        float vsq = 0.f;
        for (int c0 = 0; c0 < nch; c0 += kGrp) {
          if (!once) load(t, c0);
#pragma unroll
          for (int u = 0; u < kGrp; ++u)
            if (c0 + u < nch) {
              float ve[kEpl<T>];
#pragma unroll
              for (int e = 0; e < kEpl<T>; ++e) ve[e] = elem_of<T>(vf[u], e);
              if (g0 == 0)
#pragma unroll
                for (int e = 0; e < kEpl<T>; ++e) vsq = fmaf(ve[e], ve[e], vsq);
#pragma unroll
              for (int rb = 0; rb < kRB; ++rb) {
                const int ch = (g0 + rb) * nch + c0 + u;
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
        if (g0 == 0) vn2 = add_xor32(add_xor16(vsq));
        float sum = 0.f;
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
          const f32x4 m4 = st[(g0 + rb) * 12 + lg], r4 = st[(g0 + rb) * 12 + 4 + lg], y4 = st[(g0 + rb) * 12 + 8 + lg];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = 16 * (g0 + rb) + 4 * lg + r, m = r0 + row;
            const bool seen = m < M && t + li < nrel && k_begin + t + li <= Lk - W + dv.w.mod(m);
            float p = fminf(__builtin_amdgcn_exp2f((s[rb][r] - m4[r]) * scale_log2) * r4[r], 1.f);
            if (p_round) p = round_through<T>(p);
            const float terms = vn2 + y4[r];
            float d2 = fmaf(-2.f, gg[rb][r], terms);
            // (NaN counts as cancelled, so that infinite rows give what the
            // direct form gives.)
            uint64_t need = __ballot(seen && !(d2 >= kDirect * terms));
            while (need) {
              const int l = __builtin_ctzll(need);
              need &= need - 1;
              const T* vrow = reinterpret_cast<const T*>(vhead + (int64_t)(t + (l & 15)) * kvs.v_rb);
              const float* yrow = yrow0 + (int64_t)(16 * (g0 + rb) + 4 * (l >> 4) + r) * D;
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
        }
        total += sum;
      }
      total = add_xor16(add_xor32(total));
      if (lg == 0) {
        if (r0) total += sc[t + li];
        if (r0 + rs >= M) {
          if (t + li < nrel) scores[(int64_t)head * Lk + k_begin + t + li] = total / static_cast<float>(g);
        } else {
          sc[t + li] = total;
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
  const int CG = (D + 63) / 64, KG = part_kg(CG);
  const ScoreDiv dv{Div::of(p.n_mc), Div::of(p.s1), Div::of(Hkv), Div::of(W)};
  const size_t ops = (size_t)kRB * nch * 64 * 16;
  const bool qvec = q_sd == 1 && (q_sb * sizeof(T)) % 16 == 0 && (q_sh * sizeof(T)) % 16 == 0 &&
                    (q_ss * sizeof(T)) % 16 == 0 && (reinterpret_cast<uintptr_t>(q) & 15u) == 0;
  const size_t lds1 = std::max(ops + (size_t)16 * kRB * kPPitch * 4, (size_t)KG * 16 * kRB * (CG * 64 + 4) * 4);
  const dim3 g1(p.heads * p.n_mc * p.s1), b1(64 * kPartWaves);
  auto part = [&](auto kern, size_t lds) {
    launch(kern, g1, b1, lds, st, qq, q_sb, q_sh, q_ss, q_sd, qvec, kk, vv, kvs, Hkv, Lq, Lk, D, W, p.g, p.M, p.n_mc, p.s1,
           p.kps1, scale_log2, part_ml, part_y, row_mr, dv);
  };
  if (flash) {
    part(genm_part_kernel<T, kRB, kFlash>, lds1);
  } else {
    part(genm_part_kernel<T, kRB, kStats>, ops);
    part(genm_part_kernel<T, kRB, kSum>, lds1);
  }
  launch(genm_merge_kernel<T>, dim3(p.M, p.heads), dim3(64), 0, st, part_ml, part_y, p.n_mc, p.s1, p.M, D,
         scale_log2, flash ? 1 : 0, y_round, ystat, yf, row_mr, zero_ptr, zero_words);
  // Keys per workgroup: 64 (16 per wave) until there are more workgroups than
  // the GPU runs at once, then more, so that staging Q and Y is shared.
  constexpr int kStep = 16 * kScoreWaves;
  const int steps = (Lk + kStep - 1) / kStep;
  const int per = std::min(16, std::max(1, (int)(((int64_t)p.heads * steps + 1023) / 1024)));
  const int kpw = per * kStep, wgs = (Lk + kpw - 1) / kpw;
  // Rows staged together: all, up to half of the CU's LDS.
  constexpr size_t kStageBytes = 80 * 1024;
  auto score = [&](auto kern, size_t yv) {
    const size_t per_group = ops * (1 + yv) + 16 * kRB * 12;
    const int groups = (p.M + 16 * kRB - 1) / (16 * kRB);
    const int rs = 16 * kRB * (int)std::max<size_t>(1, std::min<size_t>(groups, kStageBytes / per_group));
    launch(kern, dim3(p.heads * wgs), dim3(64 * kScoreWaves), per_group * (rs / (16 * kRB)) + (size_t)kpw * 4, st, qq,
           q_sb, q_sh, q_ss, q_sd, qvec, kk, vv, kvs, Hkv, Lq, Lk, D, W, p.g, p.M, p.mpad, scale_log2, eps, p_round,
           kpw, rs, ystat, yf, row_mr, scores, ScoreDiv{dv.n_mc, Div::of(wgs), dv.hkv, dv.w});
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
