// Decode step on the compressed cache: append the new token's K/V row and
// attend to every stored row (dropkv_cache.py:609-617 appends with torch.cat
// and the model then runs its attention over the concatenation).
//
// The cache lives in preallocated buffers [B, Hkv, C, D] whose first n rows
// are filled; n is read from device memory, so one captured launch serves
// every step of a decode loop (the caller advances n between steps).  The
// new row is not written before the attention: the workgroup that owns key n
// takes it from the k/v inputs and stores it, and no other workgroup reads
// row n in the same launch.
//
// Two kernels: split-key partials (online softmax per query head of the GQA
// group, one workgroup per (b, kv head, key split)) and a merge over the
// splits that writes the output in the [B, 1, Hq, D] layout of the
// attention's output.
#include "dkv_common.h"
#include "dkv_internal.h"

#include <algorithm>
#include <cmath>

namespace dkv {

constexpr int kDecMaxG = 16;      // query heads per KV head: the 16 columns of the MFMA tiles
constexpr int kDecMaxSplits = 64;

struct DecodeArgs {
  const void* q;  // [B, Hq, 1, D] element strides
  int64_t q_sb, q_sh, q_sd;
  const void* kn;  // new K/V rows [B, Hkv, 1, D] element strides
  const void* vn;
  int64_t n_sb, n_sh, n_sd;
  void* kbuf;  // [B, Hkv, C, D] contiguous
  void* vbuf;
  const int* n_rows;  // rows already stored (device)
  int B, Hq, Hkv, D, C, S;
  int kps;  // rows of the buffer per split (whole tiles)
  int qvec, nvec;  // rows of q / of the new K and V as 16-byte loads
  float scale_log2;
  float* part_m;  // [B*Hkv, S, g]
  float* part_l;
  float* part_o;  // [B*Hkv, S, g, D]
  void* out;      // [B, 1, Hq, D] element strides
  int64_t o_sb, o_sh, o_sd;
};

// One wave per (b, kv head, key split).  Split s owns buffer rows
// [s * kps, (s + 1) * kps) whatever the row count, so its first tile's loads
// are issued before the count has arrived; rows past the new row n are
// masked (splits past n write empty partials).  The new row is held in
// registers, takes row n's place in its tile, and is stored into the buffer
// only after the attention, so that no wave waits on it.  Tiles of 32 keys
// (buffer views: rows past the buffer read as zeros): K in registers as the
// MFMA operand, V through LDS for the transposing reads, and the next tile's
// loads issued as soon as a tile's registers are consumed, so that a wave
// always has 16 KB on the way (D = 128).  Both products run on the matrix
// cores with the group's query heads as the 16 columns (heads past the group
// are zero): S^T = K Q^T per 16-key block, and O^T += V^T P^T per 32 keys, P in
// two parts (hi and the rounded remainder, ~16 significant bits).  Lane
// (li, lg) holds head li's logits of keys 16 kb + 4 lg + r and its outputs at
// columns 16 dt + 4 lg + r; a head's maximum and sum combine its four lanes.
//
// Bound: HBM for long caches of a batch.  With 64-key steps staged through LDS
// one after the other (32 KB a wave, five waves per CU, nothing in flight
// during a step's arithmetic, last steps of a few rows) a call with 8 x 8 heads
// of 8004 rows, D = 128 (262 MB), took 75.6 us; tiles in flight under the
// arithmetic, whole tiles per split: 50 us (5.2 TB/s).
constexpr int kDecTile = 32;

// Eight elements from d0 of a row: one 16-byte load, or by stride.
template <typename T>
__device__ __forceinline__ typename Elem<T>::v8 load8(const T* row, int d0, int64_t sd, bool vec) {
  typename Elem<T>::v8 x;
  if (vec) {
    x = *reinterpret_cast<const typename Elem<T>::v8*>(row + d0);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = row[(int64_t)(d0 + e) * sd];
  }
  return x;
}

template <typename T, int D>
__global__ void __launch_bounds__(64) decode_partial_kernel(DecodeArgs a) {
  typedef typename Elem<T>::v8 v8;
  constexpr int KK = D / 32;             // k-steps of the logits
  constexpr int DT = D / 16;             // 16-column blocks of the output
  constexpr int CPR = D / 8;             // 16-byte chunks per row
  constexpr int GRP = 64 / CPR;          // rows per load round
  constexpr int NVC = kDecTile / GRP;    // V chunks per lane and tile
  constexpr int kVPitch = D + 16;        // as pass 1's V tile: transposing reads without bank conflicts
  constexpr uint32_t kRowBytes = D * (uint32_t)sizeof(T);
  const int bh = blockIdx.x / a.S, split = blockIdx.x % a.S;
  const int b = bh / a.Hkv, hkv = bh % a.Hkv;
  const int g = a.Hq / a.Hkv;
  const int lane = threadIdx.x;
  const int li = lane & 15, lg = lane >> 4;

  __shared__ __attribute__((aligned(16))) T vt[kDecTile * kVPitch];

  T* kb = static_cast<T*>(a.kbuf) + (int64_t)bh * a.C * D;
  T* vb = static_cast<T*>(a.vbuf) + (int64_t)bh * a.C * D;
  const rsrc_t krs = make_rsrc(kb, (uint32_t)a.C * kRowBytes), vrs = make_rsrc(vb, (uint32_t)a.C * kRowBytes);
  const int k0 = split * a.kps;
  const uint32_t k_lane = li * kRowBytes + 16u * lg;
  const int v_row = lane / CPR, v_col = 8 * (lane % CPR);
  const uint32_t v_lane = v_row * kRowBytes + v_col * (uint32_t)sizeof(T);
  v8 kop[2][KK];
  u32x4 vch[NVC];
  auto load_k = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        kop[h][kk] = bitcast_u4<v8>(buf_load16(krs, k_lane + (uint32_t)(j0 + 16 * h) * kRowBytes + 64u * kk));
  };
  auto load_v = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NVC; ++i) vch[i] = buf_load16(vrs, v_lane + (uint32_t)(j0 + i * GRP) * kRowBytes);
  };
  load_k(k0);
  load_v(k0);
  const int n_in = *a.n_rows;

  // Q as the B operand: lane (li, lg) holds head li's elements 32 kk + 8 lg .. +7.
  v8 qop[KK];
  {
    const bool hv = li < g;
    const T* qh = static_cast<const T*>(a.q) + (int64_t)b * a.q_sb + (int64_t)(hkv * g + (hv ? li : 0)) * a.q_sh;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qop[kk] = load8(qh, 32 * kk + 8 * lg, a.q_sd, a.qvec);
      if (!hv) qop[kk] = v8{};
    }
  }
  // The new row, in the lanes' K operand and V chunk layouts.
  const T* kn = static_cast<const T*>(a.kn) + (int64_t)b * a.n_sb + (int64_t)hkv * a.n_sh;
  const T* vn = static_cast<const T*>(a.vn) + (int64_t)b * a.n_sb + (int64_t)hkv * a.n_sh;
  v8 kx[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) kx[kk] = load8(kn, 32 * kk + 8 * lg, a.n_sd, a.nvec);
  const v8 vx = load8(vn, v_col, a.n_sd, a.nvec);
  const int n = min(n_in, a.C - 1);  // the host keeps n < C; the clamp keeps every access in bounds
  const int k1 = min(k0 + a.kps, n + 1);
  const bool own_n = k0 <= n && n < k1;  // this split holds the new row

  // Head li, log2 units; lsum is this lane's share.  The maximum starts finite, so
  // that logits of -inf get no weight (-inf - -inf would be NaN) where a tile or
  // the whole split has no other.
  float m = -__FLT_MAX__, lsum = 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tr_row = 4 * lg + li / 4, tr_col = 4 * (li % 4);

  for (int j0 = k0; j0 < k1; j0 += kDecTile) {
    if (own_n && n < j0 + kDecTile) {
      // The last tile, up to row n: the new row in its place, and V rows past
      // it to zero (their p is 0, but 0 * NaN is not, and those rows hold
      // whatever the buffer held).
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
          if (j0 + 16 * h + li == n) kop[h][kk] = kx[kk];
#pragma unroll
      for (int i = 0; i < NVC; ++i) {
        const int row = j0 + v_row + i * GRP;
        if (row == n) vch[i] = __builtin_bit_cast(u32x4, vx);
        if (row > n) vch[i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
    // S^T = K Q^T, 16 keys per block; then the K registers are free.
    f32x4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) acc = Elem<T>::mfma(kop[h][kk], qop[kk], acc);
      s[h] = acc;
    }
    load_k(j0 + kDecTile);
#pragma unroll
    for (int i = 0; i < NVC; ++i)
      *reinterpret_cast<u32x4*>(vt + (v_row + i * GRP) * kVPitch + v_col) = vch[i];
    load_v(j0 + kDecTile);
    // Keys past the split's last one masked; the head's tile maximum over
    // its four lanes (IEEE maximum; scaling by a positive factor keeps the
    // order).
    const int nb = k1 - j0;
    float tmax = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = (16 * h + 4 * lg + r) < nb ? s[h][r] : -INFINITY;
        s[h][r] = x;
        tmax = __builtin_elementwise_maximum(tmax, x);
      }
    tmax = max_xor32(max_xor16(tmax)) * a.scale_log2;
    const float mnew = fmaxf(m, tmax);
    const float alpha = __builtin_amdgcn_exp2f(m - mnew);
    // P^T operand: element e is key 4 lg + e (e < 4) or 16 + 4 lg + e - 4; the
    // transposing V reads below give V^T in that key order.
    float psum = 0.f;
    v8 phi, plo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = __builtin_amdgcn_exp2f(fmaf(s[e / 4][e % 4], a.scale_log2, -mnew));
      psum += x;
      phi[e] = static_cast<T>(x);
      plo[e] = static_cast<T>(x - static_cast<float>(phi[e]));
    }
    lsum = lsum * alpha + psum;
    m = mnew;
    if (wave_any(alpha != 1.f))
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    // O^T += V^T P^T: lane (li, lg) of the A operand needs V[key][16 dt + li]
    // for the eight keys above; a transposing read gives output lane i of
    // each 16-lane group element e of input lane 4e + i/4's 8 bytes, element
    // i % 4, so input lane li reads key base + li/4, columns
    // 16 dt + 4 (li % 4) .. +3.
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      typedef short s4 __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) s4 lds_s4;
      const s4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + tr_row * kVPitch + 16 * dt + tr_col));
      const s4 x1 =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + (16 + tr_row) * kVPitch + 16 * dt + tr_col));
      const v8 aop = __builtin_bit_cast(v8, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
      o[dt] = Elem<T>::mfma(aop, phi, o[dt]);
      o[dt] = Elem<T>::mfma(aop, plo, o[dt]);
    }
  }

  if (own_n)  // store the new row
    for (int d = lane; d < D; d += 64) {
      kb[(int64_t)n * D + d] = kn[(int64_t)d * a.n_sd];
      vb[(int64_t)n * D + d] = vn[(int64_t)d * a.n_sd];
    }
  // The split's partials (heads h < g).
  lsum = add_xor32(add_xor16(lsum));
  const int64_t base = ((int64_t)bh * a.S + split) * g;
  if (li < g) {
    float* po = a.part_o + (base + li) * D + 4 * lg;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(po + 16 * dt) = o[dt];
    if (lg == 0) {
      a.part_m[base + li] = m;
      a.part_l[base + li] = lsum;
    }
  }
}

// One wave per query head: combine the splits and write the output row.
// Lane s holds split s's (m, l); the partial outputs, 16 bytes a lane and so
// two (D = 128) or four (D = 64) splits per load, are all issued together with
// the statistics, before the reductions: one round trip whatever the number
// of splits.  (One element a lane in batches of 32 splits took a second round
// trip past 32: 12.8 against 11.5 us per layer, both kernels, at 57 splits of
// 3300 rows, 32 query and 8 KV heads of 128.)
template <typename T, int D>
__global__ void __launch_bounds__(64) decode_merge_kernel(DecodeArgs a) {
  constexpr int LPR = D / 4;                  // lanes per row
  constexpr int SPL = 64 / LPR;               // splits per load
  constexpr int NL = kDecMaxSplits / SPL;     // loads
  const int g = a.Hq / a.Hkv;
  const int b = blockIdx.x / a.Hq, hq = blockIdx.x % a.Hq;
  const int hkv = hq / g, h = hq % g;
  const int lane = threadIdx.x;
  const int sub = lane / LPR, d0 = 4 * (lane % LPR);
  const int64_t base = ((int64_t)(b * a.Hkv + hkv) * a.S) * g + h;
  const float ml = lane < a.S ? a.part_m[base + (int64_t)lane * g] : -INFINITY;
  const float ll = lane < a.S ? a.part_l[base + (int64_t)lane * g] : 0.f;
  // (Splits past the last read as zeros.)
  const rsrc_t ors = make_rsrc(a.part_o + base * D, ((uint32_t)(a.S - 1) * g + 1) * D * 4u);
  f32x4 ob[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i)
    ob[i] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(ors, ((uint32_t)(SPL * i + sub) * g * D + d0) * 4u, 0, 0));
  const float mx = wave_max_dpp(ml);
  // Lanes past S (-inf), and splits with no rows or none above -inf, weigh 0.
  const float f = __builtin_amdgcn_exp2f(ml - mx);
  const float l = wave_sum_dpp(ll * f);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NL; ++i)
    if (i * SPL < a.S) {
      const float fs = __shfl(f, SPL * i + sub);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(fs, ob[i][e], acc[e]);
    }
  const float inv = 1.f / l;  // (0 / 0 = NaN where every logit is -inf, as softmax gives)
  T* out = static_cast<T*>(a.out) + (int64_t)b * a.o_sb + (int64_t)hq * a.o_sh;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float y = add_xor32(acc[e]);
    if (SPL == 4) y = add_xor16(y);
    if (sub == 0) out[(int64_t)(d0 + e) * a.o_sd] = static_cast<T>(y * inv);
  }
}

// Splits of a cache of C rows for `heads` (b, kv head) pairs: whole tiles, and
// no more waves than keep the memory busy, since each split also costs its
// prologue, its epilogue and D floats per query head for the merge to read
// (64 heads of 8004 rows, D = 128, both kernels: 50.1 us with 512 waves, 52.7
// with 1024, 56.1 with 2048), two tiles a split at least (a short cache of 1639
// rows, 2 heads, D = 64: 7.0 us a layer, against 8.7 with one tile a split and
// 7.7 with four).
// Where the heads do not divide the 512 waves, rounding down leaves some out.
// At D = 128 (16 KB in flight a wave) that costs less than the last, partly
// filled wave of rounding up (171 heads of 8128 rows: 124 us with 2 splits, 143
// with 3; 257 heads: 215 with 1, 219 with 2).  At D = 64 a wave has only 8 KB in
// flight, and with a sixteenth of the waves missing or more rounding up is the
// faster one (66 heads of 16320 rows: 51.4 us with 7 splits, 46.6 with 8; 171
// heads of 8128: 92 and 69; 257: 162 and 99; 384: 178 and 138; 450 heads of
// 7300: 166 and 145).
constexpr int kDecWaves = 512;
constexpr int kDecMinTiles = 2;

struct DecodeSplits {
  int S, kps;
};
static DecodeSplits decode_splits(int64_t heads, int D, int C) {
  const int tiles = (C + kDecTile - 1) / kDecTile;
  int64_t waves_per_head = kDecWaves / heads;
  if (D == 64 && heads * waves_per_head < kDecWaves - kDecWaves / 16) ++waves_per_head;
  const int want = (int)std::max<int64_t>(1, std::min<int64_t>(kDecMaxSplits, waves_per_head));
  const int per = std::max((tiles + want - 1) / want, std::min(tiles, kDecMinTiles));
  return DecodeSplits{(tiles + per - 1) / per, per * kDecTile};
}

// For the most splits that decode_splits gives any number of heads (two tiles a
// split at least), so that the size grows with the batch and the capacity: a
// workspace for the largest call holds every smaller one, whose splits may be
// more.
size_t decode_workspace_bytes(int B, int Hq, int Hkv, int D, int C) {
  const size_t tiles = ((size_t)C + kDecTile - 1) / kDecTile;
  const size_t S = std::min<size_t>(kDecMaxSplits, (tiles + kDecMinTiles - 1) / kDecMinTiles);
  const size_t rows = (size_t)B * Hkv * S * (Hq / Hkv);
  return rows * sizeof(float) * (2 + (size_t)D) + 256;
}

template <typename T, int D>
static hipError_t launch_decode_t(DecodeArgs a, hipStream_t st) {
  const int g = a.Hq / a.Hkv;
  if (g < 1 || g > kDecMaxG) return hipErrorInvalidValue;
  const dim3 grid(a.B * a.Hkv * a.S);
  launch((decode_partial_kernel<T, D>), grid, dim3(64), 0, st, a);
  launch((decode_merge_kernel<T, D>), dim3(a.B * a.Hq), dim3(64), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_decode_attention(const DecodeParams& p, hipStream_t st) {
  DecodeArgs a;
  a.q = p.q;
  a.q_sb = p.q_sb;
  a.q_sh = p.q_sh;
  a.q_sd = p.q_sd;
  a.kn = p.kn;
  a.vn = p.vn;
  a.n_sb = p.n_sb;
  a.n_sh = p.n_sh;
  a.n_sd = p.n_sd;
  a.kbuf = p.kbuf;
  a.vbuf = p.vbuf;
  a.n_rows = p.n_rows;
  a.B = p.B;
  a.Hq = p.Hq;
  a.Hkv = p.Hkv;
  a.D = p.D;
  a.C = p.C;
  const DecodeSplits sp = decode_splits((int64_t)p.B * p.Hkv, p.D, p.C);
  a.S = sp.S;
  a.kps = sp.kps;
  a.scale_log2 = p.scale * 1.4426950408889634f;
  const size_t rows = (size_t)p.B * p.Hkv * a.S * (p.Hq / p.Hkv);
  char* ws = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(p.workspace) + 15) & ~(uintptr_t)15);
  auto vec = [](const void* x, int64_t sb, int64_t sh, int64_t sd) {
    return (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && sd == 1 && sb % 8 == 0 && sh % 8 == 0;
  };
  a.qvec = vec(p.q, p.q_sb, p.q_sh, p.q_sd);
  a.nvec = vec(p.kn, p.n_sb, p.n_sh, p.n_sd) && vec(p.vn, p.n_sb, p.n_sh, p.n_sd);
  a.part_m = reinterpret_cast<float*>(ws);
  a.part_l = a.part_m + rows;
  a.part_o = a.part_m + ((2 * rows + 3) & ~(size_t)3);  // 16-byte stores
  a.out = p.out;
  a.o_sb = p.o_sb;
  a.o_sh = p.o_sh;
  a.o_sd = p.o_sd;
  if (p.dtype_bf16) {
    if (p.D == 64) return launch_decode_t<__bf16, 64>(a, st);
    return launch_decode_t<__bf16, 128>(a, st);
  }
  if (p.D == 64) return launch_decode_t<_Float16, 64>(a, st);
  return launch_decode_t<_Float16, 128>(a, st);
}

}  // namespace dkv
