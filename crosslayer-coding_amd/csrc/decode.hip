// Sparse cross-layer decode, decoder repacking, densify and decoder norms.
//
// Decode (reference clt/models/decoder.py:176-340): the reference multiplies dense
// [T,F] activations that are >99 % zeros by every decoder.  Here each (token, target)
// pair is one wavefront that walks the survivor rows of the sources s <= t, fetches the
// decoder vector of every active feature (feature-major packing: one contiguous
// d-element run, 16 bytes per lane per load) and accumulates in fp32 registers; the
// output row is written once.
#include <cmath>
#include <type_traits>
#include "clt_common.h"

namespace {

// Row layout seen by one wavefront: NF full chunks of 64 lanes x 16 bytes, then an optional
// tail chunk - TAIL 1: 64 lanes x 8 bytes (exactly fills the row), TAIL 2: a 16-byte chunk
// in which only the leading lanes are inside the row.
template <typename T> struct WVec;
template <> struct WVec<float> {
  static constexpr int V = 4;   // elements per 16 bytes
  __device__ static __forceinline__ void fma16(float *acc, const uint4 &w, float v) {
    acc[0] = fmaf(v, __uint_as_float(w.x), acc[0]); acc[1] = fmaf(v, __uint_as_float(w.y), acc[1]);
    acc[2] = fmaf(v, __uint_as_float(w.z), acc[2]); acc[3] = fmaf(v, __uint_as_float(w.w), acc[3]);
  }
  __device__ static __forceinline__ void fma8(float *acc, const uint2 &w, float v) {
    acc[0] = fmaf(v, __uint_as_float(w.x), acc[0]); acc[1] = fmaf(v, __uint_as_float(w.y), acc[1]);
  }
};
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;

template <> struct WVec<bf16_t> {
  static constexpr int V = 8;
  // Two survivors at once: for each pair of bf16 weights in a 32-bit word, a byte permute puts
  // the same element of both rows side by side and v_dot2c_f32_bf16 multiplies them with the two
  // activation values (bf16 pair `vv`) and accumulates in fp32 - one op per element instead of two.
  // `vp`: the two activation values as raw 16-bit elements, (first | second << 16)
  __device__ static __forceinline__ void dot32(float *acc, uint32_t a, uint32_t b, uint32_t vp) {
    const bf16x2_t vv = __builtin_bit_cast(bf16x2_t, vp);
    const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05040100u);   // (a.lo16, b.lo16)
    const uint32_t hi = __builtin_amdgcn_perm(b, a, 0x07060302u);   // (a.hi16, b.hi16)
    acc[0] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, lo), vv, acc[0], false);
    acc[1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, hi), vv, acc[1], false);
  }
  __device__ static __forceinline__ void dot16(float *acc, const uint4 &a, const uint4 &b, uint32_t vp) {
    dot32(acc, a.x, b.x, vp); dot32(acc + 2, a.y, b.y, vp); dot32(acc + 4, a.z, b.z, vp); dot32(acc + 6, a.w, b.w, vp);
  }
  __device__ static __forceinline__ void dot8(float *acc, const uint2 &a, const uint2 &b, uint32_t vp) {
    dot32(acc, a.x, b.x, vp); dot32(acc + 2, a.y, b.y, vp);
  }
  __device__ static __forceinline__ void fma32(float *acc, uint32_t u, float v) {
    acc[0] = fmaf(v, __uint_as_float(u << 16), acc[0]);
    acc[1] = fmaf(v, __uint_as_float(u & 0xFFFF0000u), acc[1]);
  }
  __device__ static __forceinline__ void fma16(float *acc, const uint4 &w, float v) {
    fma32(acc, w.x, v); fma32(acc + 2, w.y, v); fma32(acc + 4, w.z, v); fma32(acc + 6, w.w, v);
  }
  __device__ static __forceinline__ void fma8(float *acc, const uint2 &w, float v) {
    fma32(acc, w.x, v); fma32(acc + 2, w.y, v);
  }
};

// IEEE half: the same scheme with v_dot2_f32_f16 (exact products, fp32 accumulation)
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
template <> struct WVec<f16_t> {
  static constexpr int V = 8;
  __device__ static __forceinline__ void dot32(float *acc, uint32_t a, uint32_t b, uint32_t vp) {
    const f16x2_t vv = __builtin_bit_cast(f16x2_t, vp);
    const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05040100u);
    const uint32_t hi = __builtin_amdgcn_perm(b, a, 0x07060302u);
    acc[0] = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, lo), vv, acc[0], false);
    acc[1] = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, hi), vv, acc[1], false);
  }
  __device__ static __forceinline__ void dot16(float *acc, const uint4 &a, const uint4 &b, uint32_t vp) {
    dot32(acc, a.x, b.x, vp); dot32(acc + 2, a.y, b.y, vp); dot32(acc + 4, a.z, b.z, vp); dot32(acc + 6, a.w, b.w, vp);
  }
  __device__ static __forceinline__ void dot8(float *acc, const uint2 &a, const uint2 &b, uint32_t vp) {
    dot32(acc, a.x, b.x, vp); dot32(acc + 2, a.y, b.y, vp);
  }
  __device__ static __forceinline__ void fma32(float *acc, uint32_t u, float v) {
    float lo, hi;
    unpack_pair<f16_t>(u, lo, hi);
    acc[0] = fmaf(v, lo, acc[0]);
    acc[1] = fmaf(v, hi, acc[1]);
  }
  __device__ static __forceinline__ void fma16(float *acc, const uint4 &w, float v) {
    fma32(acc, w.x, v); fma32(acc + 2, w.y, v); fma32(acc + 4, w.z, v); fma32(acc + 6, w.w, v);
  }
  __device__ static __forceinline__ void fma8(float *acc, const uint2 &w, float v) {
    fma32(acc, w.x, v); fma32(acc + 2, w.y, v);
  }
};

__device__ __forceinline__ int64_t decoder_slot(int tying, int64_t s, int64_t t, int64_t L) {
  if (tying == CLT_TYING_PER_SOURCE) return s;
  if (tying == CLT_TYING_PER_TARGET) return t;
  return s * L - (s * (s - 1)) / 2 + (t - s);
}

static inline int64_t decoder_slot_host(int tying, int64_t s, int64_t t, int64_t L) {
  if (tying == CLT_TYING_PER_SOURCE) return s;
  if (tying == CLT_TYING_PER_TARGET) return t;
  return s * L - (s * (s - 1)) / 2 + (t - s);
}

// UU decoder vectors in flight: the row pieces of one lane plus the (wave-uniform) weights.
template <typename T, int NF, int TAIL, int UU> struct RowBatch {
  uint4 wq[UU][NF > 0 ? NF : 1];
  uint4 wt16[UU];
  uint2 wt8[UU];
  float v[UU];

  // request rows i0 .. i0+UU-1 of the 64 survivors held one per lane in (my_col, my_val)
  __device__ __forceinline__ void load(const T *wbase, int64_t d, int32_t my_col, float my_val, int i0, int n,
                                       int lane, int64_t tail_off, bool tail_on) {
    constexpr int V = WVec<T>::V;
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      const int idx = (i0 + u) < n ? (i0 + u) : (n - 1);   // clamp: a repeated fetch, weight 0
      const int32_t f = __builtin_amdgcn_readlane(my_col, idx);
      const float vv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_val), idx));
      v[u] = (i0 + u) < n ? vv : 0.0f;
      const T *wrow = wbase + (int64_t)f * d;
#pragma unroll
      for (int c = 0; c < NF; ++c) wq[u][c] = *reinterpret_cast<const uint4 *>(wrow + (int64_t)c * 64 * V + (int64_t)lane * V);
      if (TAIL == 1) wt8[u] = *reinterpret_cast<const uint2 *>(wrow + tail_off);
      if (TAIL == 2) wt16[u] = tail_on ? *reinterpret_cast<const uint4 *>(wrow + tail_off) : make_uint4(0, 0, 0, 0);
    }
  }

  __device__ __forceinline__ void consume(float *acc) const {
    constexpr int V = WVec<T>::V;
    if constexpr (sizeof(T) == 2 && (UU % 2) == 0) {
      // bf16: the activation values are exact bf16 numbers, so two of them fit one dot2 operand
#pragma unroll
      for (int u = 0; u < UU; u += 2) {
        const uint32_t vv = raw16_of<T>(v[u]) | (raw16_of<T>(v[u + 1]) << 16);
#pragma unroll
        for (int c = 0; c < NF; ++c) WVec<T>::dot16(acc + c * V, wq[u][c], wq[u + 1][c], vv);
        if (TAIL == 1) WVec<T>::dot8(acc + NF * V, wt8[u], wt8[u + 1], vv);
        if (TAIL == 2) WVec<T>::dot16(acc + NF * V, wt16[u], wt16[u + 1], vv);
      }
    } else {
#pragma unroll
      for (int u = 0; u < UU; ++u) {
#pragma unroll
        for (int c = 0; c < NF; ++c) WVec<T>::fma16(acc + c * V, wq[u][c], v[u]);
        if (TAIL == 1) WVec<T>::fma8(acc + NF * V, wt8[u], v[u]);
        if (TAIL == 2) WVec<T>::fma16(acc + NF * V, wt16[u], v[u]);
      }
    }
  }
};

// Fetch UU decoder vectors (all requests issued before the first multiply) and accumulate.
template <typename T, int NF, int TAIL, int UU>
__device__ __forceinline__ void decode_batch(float *acc, const T *wbase, int64_t d, int32_t my_col, float my_val,
                                             int i0, int n, int lane, int64_t tail_off, bool tail_on) {
  RowBatch<T, NF, TAIL, UU> rb;
  rb.load(wbase, d, my_col, my_val, i0, n, lane, tail_off, tail_on);
  rb.consume(acc);
}

// Up to 64 survivors (one per lane) with two batches in flight: while one batch is multiplied
// the next one is already on its way.
template <typename T, int NF, int TAIL, int UU>
__device__ __forceinline__ void decode_chunk_pipelined(float *acc, const T *wbase, int64_t d, int32_t my_col,
                                                       float my_val, int n, int lane, int64_t tail_off, bool tail_on) {
  RowBatch<T, NF, TAIL, UU> ra, rb;
  ra.load(wbase, d, my_col, my_val, 0, n, lane, tail_off, tail_on);
  for (int i0 = 0; i0 < n; i0 += 2 * UU) {
    if (i0 + UU < n) rb.load(wbase, d, my_col, my_val, i0 + UU, n, lane, tail_off, tail_on);
    ra.consume(acc);
    if (i0 + UU < n) {
      if (i0 + 2 * UU < n) ra.load(wbase, d, my_col, my_val, i0 + 2 * UU, n, lane, tail_off, tail_on);
      rb.consume(acc);
    }
  }
}

// The partial rows are touched once per launch: streaming loads / stores keep them from pushing the
// decoder slice out of the L2.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ldg_stream4(const float *p) {
  const f32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t *>(p));
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void stg_stream4(float *p, float4 v) {
  f32x4_t q = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(q, reinterpret_cast<f32x4_t *>(p));
}

template <typename T, int NF, int TAIL, bool SLICED> constexpr int decode_min_waves() {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int nacc = NF * V + (TAIL == 1 ? V / 2 : TAIL == 2 ? V : 0);
  return (SLICED && sizeof(T) == 2 && nacc <= 12) ? 4 : 1;
}

constexpr int SLICED_NTOK = 4;   // tokens per wavefront in the sliced kernel
// Launches of at most DECODE_FEW (target, token) rows, a wavefront for each SIMD: nothing but a row's own loads hides their
// latency, so 16 survivors are asked for at once, and every row has a workgroup, and so an L1, to itself.
// L = 3, d = 768, float32, 32 tokens x 16 survivors: 33.6 -> 19.9 us; a forward waited for 176 -> 165 us, L = 2, d = 512, 500
// tokens 304 -> 291 us.  Above the line a SIMD has several rows to switch between, and 16 in flight cost wavefronts; rows of
// more than four registers' worth of pieces (NF = 4) would need 320 registers for them.  In bf16 three pieces and a half one
// (d = 1792) are kept to 8 in flight: at 16 they need 19 registers more than there are, and every survivor pays for moving
// them.  L = 4, 32 tokens x 100, us, launch of many rows / this: d = 1536 bf16 70 / 46, fp16 88 / 45; d = 1792 bf16 75 / 58 (143
// at 16), fp16 91 / 49; d = 2000 78 / 61; d = 896 float32 80 / 50.
constexpr int DECODE_FEW = 1024, DECODE_FEW_U = 16;
template <typename T, int NF, int TAIL> constexpr int decode_few_in_flight() {
  return std::is_same<T, bf16_t>::value && NF == 3 && TAIL == 1 ? 8 : DECODE_FEW_U;
}

// One wavefront per (target, token): walks all sources s <= t, accumulates in registers,
// writes the output row once.  Used for small batches.
//
// SLICED (large batches): one launch per source layer `src`; one wavefront per
// (target >= src, token, feature slice).  The feature axis is cut into `ns` slices and block b
// works on slice b % ns.  Workgroups are handed to the XCDs round-robin, so with ns = 8 each
// XCD sees one slice of a decoder matrix (1/8 of its rows); blocks are ordered target-major,
// so at any moment the wavefronts resident on an XCD gather from ONE slice of ONE matrix
// (a few MB, L2-resident) while all tokens stream past - every row is fetched from HBM once
// and then hit ~T*k/F times in L2.  The price is that a (target, token, slice) accumulator
// cannot stay in registers across launches: it lives as an fp32 partial row that each launch
// reads, updates and writes back (skipped when the token has no survivor in the slice).
// k_decode_reduce finally adds the slices in a fixed order and applies bias / skip / rounding.
template <typename T, int NF, int TAIL, int U, bool AFFINE, bool SLICED>
// The sliced variant with up to 12 accumulators per lane (d <= 768 in bf16) needs 129 registers when left
// alone, one more than four wavefronts per SIMD allow; held to 128 it spills nothing and runs 4 % faster.
// Wider rows would spill at that limit and keep the compiler's own choice.
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(decode_min_waves<T, NF, TAIL, SLICED>(), 8))) void k_decode(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col, const T *__restrict__ val,
    const T *__restrict__ wp, const float *__restrict__ bias_sum, const T *__restrict__ foff,
    const T *__restrict__ fscale, const float *__restrict__ skip_add, void *__restrict__ out,
    int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin, int64_t t_end,
    uint64_t src_mask, int out_f32, const int32_t *__restrict__ sptr, float *__restrict__ partial, int ns,
    int src, int64_t pitch) {
  constexpr int V = WVec<T>::V;
  constexpr int HV = V / 2;                       // elements per 8 bytes
  constexpr int NACC = NF * V + (TAIL == 1 ? HV : TAIL == 2 ? V : 0);
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int64_t tok_per_blk = SLICED ? (int64_t)nwv * SLICED_NTOK : (int64_t)nwv;
  const int64_t blocks_per_t = (Tn + tok_per_blk - 1) / tok_per_blk;
  const int64_t bid = SLICED ? (int64_t)blockIdx.x / ns : (int64_t)blockIdx.x;
  const int slice = SLICED ? (int)(blockIdx.x % ns) : 0;
  // single pass: heaviest targets (most sources) first; sliced: targets in ascending order
  const int64_t t = SLICED ? t_begin + bid / blocks_per_t : t_end - 1 - bid / blocks_per_t;
  const int64_t tok = (bid % blocks_per_t) * nwv + wv;
  if (!SLICED && tok >= Tn) return;
  float acc[NACC];
#pragma unroll
  for (int j = 0; j < NACC; ++j) acc[j] = 0.0f;
  const int64_t tail_off = TAIL == 1 ? (int64_t)NF * 64 * V + (int64_t)lane * HV : (int64_t)NF * 64 * V + (int64_t)lane * V;
  const bool tail_on = TAIL == 1 ? true : (TAIL == 2 ? tail_off < d : false);

  auto gather_rows = [&](int64_t s, int32_t b, int32_t e) {
    const T *wbase = wp + decoder_slot(tying, s, t, L) * F * pitch;
    for (int32_t j0 = b; j0 < e; j0 += 64) {
      const int n = (e - j0) < 64 ? (e - j0) : 64;
      int32_t my_col = 0; float my_val = 0.0f;
      if (lane < n) {
        my_col = col[j0 + lane];
        my_val = Elem<T>::to_f32(val[j0 + lane]);
        if (AFFINE && my_val != 0.0f) {
          if (foff) my_val = Elem<T>::round(my_val + Elem<T>::to_f32(foff[t * F + my_col]));
          if (fscale) my_val = Elem<T>::round(my_val * Elem<T>::to_f32(fscale[t * F + my_col]));
        }
      }
      int i0 = 0;
      for (; i0 + U <= n; i0 += U) decode_batch<T, NF, TAIL, U>(acc, wbase, pitch, my_col, my_val, i0, n, lane, tail_off, tail_on);
      if constexpr (U == DECODE_FEW_U) {
        for (; i0 + 4 <= n; i0 += 4) decode_batch<T, NF, TAIL, 4>(acc, wbase, pitch, my_col, my_val, i0, n, lane, tail_off, tail_on);
      }
      for (; i0 < n; i0 += 2) decode_batch<T, NF, TAIL, 2>(acc, wbase, pitch, my_col, my_val, i0, n, lane, tail_off, tail_on);
    }
  };

  if (SLICED) {
    // this wavefront: tokens tok*NTOK .. +NTOK-1 of source `src`, slice `slice`, target t.
    // Their slice bounds are fetched at once (one lane per token), and the survivor list of the
    // next token is requested before the current token's rows are gathered.
    const int64_t tok0 = tok * SLICED_NTOK;
    if (tok0 >= Tn) return;
    if (src < 0) {
      // All sources in one launch (decoders tied per target: every source <= t gathers from the same
      // matrix W[t], so the slice an XCD works on stays the same while the sources go by): the
      // accumulators stay in registers over the sources and the partial row is written once.
      const T *wb = wp + decoder_slot(tying, 0, t, L) * F * pitch;
      for (int i = 0; i < SLICED_NTOK; ++i) {
        if (tok0 + i >= Tn) break;
#pragma unroll
        for (int j = 0; j < NACC; ++j) acc[j] = 0.0f;
        for (int64_t s = 0; s <= t; ++s) {
          if (!((src_mask >> s) & 1ull)) continue;
          const int64_t r = s * Tn + tok0 + i;
          const int32_t b = sptr[r * (ns + 1) + slice], e = sptr[r * (ns + 1) + slice + 1];
          for (int32_t j0 = b; j0 < e; j0 += 64) {
            const int n = (e - j0) < 64 ? (e - j0) : 64;
            int32_t my_col = 0; float my_val = 0.0f;
            if (lane < n) { my_col = col[j0 + lane]; my_val = Elem<T>::to_f32(val[j0 + lane]); }
            if (AFFINE && my_val != 0.0f) {
              if (foff) my_val = Elem<T>::round(my_val + Elem<T>::to_f32(foff[t * F + my_col]));
              if (fscale) my_val = Elem<T>::round(my_val * Elem<T>::to_f32(fscale[t * F + my_col]));
            }
            decode_chunk_pipelined<T, NF, TAIL, (U > 6 ? 6 : U)>(acc, wb, pitch, my_col, my_val, n, lane, tail_off, tail_on);
          }
        }
        float *prow = partial + (((int64_t)slice * L + t) * Tn + tok0 + i) * d;
#pragma unroll
        for (int c = 0; c < NF; ++c) {
          float *pp = prow + (int64_t)c * 64 * V + (int64_t)lane * V;
#pragma unroll
          for (int j = 0; j < V; j += 4)
            stg_stream4(pp + j, make_float4(acc[c * V + j], acc[c * V + j + 1], acc[c * V + j + 2], acc[c * V + j + 3]));
        }
        if (TAIL == 1) {
#pragma unroll
          for (int j = 0; j < HV; ++j) prow[tail_off + j] = acc[NF * V + j];
        }
        if (TAIL == 2 && tail_on) {
#pragma unroll
          for (int j = 0; j < V; ++j) prow[tail_off + j] = acc[NF * V + j];
        }
      }
      return;
    }
    const uint64_t below = src_mask & ((1ull << src) - 1ull);
    const bool first = below == 0;   // the first source initialises the partial rows
    int32_t mb = 0, me = 0;
    if (lane < SLICED_NTOK && tok0 + lane < Tn) {
      const int64_t r = (int64_t)src * Tn + tok0 + lane;
      mb = sptr[r * (ns + 1) + slice];
      me = sptr[r * (ns + 1) + slice + 1];
    }
    const T *wbase = wp + decoder_slot(tying, src, t, L) * F * pitch;
    int32_t nb = __builtin_amdgcn_readlane(mb, 0), ne = __builtin_amdgcn_readlane(me, 0);
    int32_t nxt_col = 0; T nxt_val = Elem<T>::from_raw(0u);
    if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
#pragma unroll
    for (int i = 0; i < SLICED_NTOK; ++i) {
      const int32_t b = nb, e = ne;
      const int32_t cur_col = nxt_col; const T cur_val = nxt_val;
      if (i + 1 < SLICED_NTOK) {
        nb = __builtin_amdgcn_readlane(mb, i + 1); ne = __builtin_amdgcn_readlane(me, i + 1);
        nxt_col = 0; nxt_val = Elem<T>::from_raw(0u);
        if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
      }
      if (tok0 + i >= Tn) break;
      if (b == e && !first) continue;
      float *prow = partial + (((int64_t)slice * L + t) * Tn + tok0 + i) * d;
      float old[NACC];
#pragma unroll
      for (int j = 0; j < NACC; ++j) { old[j] = 0.0f; acc[j] = 0.0f; }
      if (!first) {   // requested before the gathers so that its latency hides behind them
#pragma unroll
        for (int c = 0; c < NF; ++c) {
          const float *pp = prow + (int64_t)c * 64 * V + (int64_t)lane * V;
#pragma unroll
          for (int j = 0; j < V; j += 4) {
            float4 q = ldg_stream4(pp + j);
            old[c * V + j] = q.x; old[c * V + j + 1] = q.y; old[c * V + j + 2] = q.z; old[c * V + j + 3] = q.w;
          }
        }
        if (TAIL == 1) {
#pragma unroll
          for (int j = 0; j < HV; ++j) old[NF * V + j] = prow[tail_off + j];
        }
        if (TAIL == 2 && tail_on) {
#pragma unroll
          for (int j = 0; j < V; ++j) old[NF * V + j] = prow[tail_off + j];
        }
      }
      for (int32_t j0 = b; j0 < e; j0 += 64) {
        const int n = (e - j0) < 64 ? (e - j0) : 64;
        int32_t my_col = cur_col; float my_val = Elem<T>::to_f32(cur_val);
        if (j0 > b) {   // more than 64 survivors in this slice: fetch the next 64
          my_col = 0; my_val = 0.0f;
          if (lane < n) { my_col = col[j0 + lane]; my_val = Elem<T>::to_f32(val[j0 + lane]); }
        }
        if (AFFINE && my_val != 0.0f) {
          if (foff) my_val = Elem<T>::round(my_val + Elem<T>::to_f32(foff[t * F + my_col]));
          if (fscale) my_val = Elem<T>::round(my_val * Elem<T>::to_f32(fscale[t * F + my_col]));
        }
        decode_chunk_pipelined<T, NF, TAIL, (U > 6 ? 6 : U)>(acc, wbase, pitch, my_col, my_val, n, lane, tail_off, tail_on);
      }
#pragma unroll
      for (int c = 0; c < NF; ++c) {
        float *pp = prow + (int64_t)c * 64 * V + (int64_t)lane * V;
#pragma unroll
        for (int j = 0; j < V; j += 4)
          stg_stream4(pp + j, make_float4(old[c * V + j] + acc[c * V + j], old[c * V + j + 1] + acc[c * V + j + 1],
                                          old[c * V + j + 2] + acc[c * V + j + 2], old[c * V + j + 3] + acc[c * V + j + 3]));
      }
      if (TAIL == 1) {
#pragma unroll
        for (int j = 0; j < HV; ++j) prow[tail_off + j] = old[NF * V + j] + acc[NF * V + j];
      }
      if (TAIL == 2 && tail_on) {
#pragma unroll
        for (int j = 0; j < V; ++j) prow[tail_off + j] = old[NF * V + j] + acc[NF * V + j];
      }
    }
    return;
  }

  // the token's lists of all sources, a lane each: their places arrive together
  int32_t my_b = 0, my_e = 0;
  if (lane <= t) { my_b = row_ptr[lane * Tn + tok]; my_e = row_ptr[lane * Tn + tok + 1]; }
  for (int s = 0; s <= (int)t; ++s) {
    if (!((src_mask >> s) & 1ull)) continue;
    gather_rows(s, __builtin_amdgcn_readlane(my_b, s), __builtin_amdgcn_readlane(my_e, s));
  }
  // epilogue: bias, skip term, one write of the output row
  auto emit = [&](int64_t o, const float *a, int cnt, bool on) {
    if (!on) return;
    for (int j = 0; j < cnt; ++j) {
      float y = a[j];
      if (bias_sum) y += bias_sum[t * d + o + j];
      if (skip_add) y += skip_add[(t * Tn + tok) * d + o + j];
      if (out_f32) ((float *)out)[(t * Tn + tok) * d + o + j] = y;
      else ((T *)out)[(t * Tn + tok) * d + o + j] = Elem<T>::from_f32(y);
    }
  };
#pragma unroll
  for (int c = 0; c < NF; ++c) emit((int64_t)c * 64 * V + (int64_t)lane * V, acc + c * V, V, true);
  if (TAIL == 1) emit(tail_off, acc + NF * V, HV, true);
  if (TAIL == 2) emit(tail_off, acc + NF * V, V, tail_on);
}

// How the units (slice, column part) of one target are dealt to the 8 XCDs: `full` rounds in which XCD x
// takes unit round * 8 + x over all tokens, then the `rem` units that are left over, with the tokens of each
// split between q XCDs so that all eight stay busy (rem divides 8: one round, q = 8 / rem; otherwise `rem`
// rounds in which all XCDs share one unit, q = 8).  Blocks go to the XCDs round-robin, so block b runs on
// XCD b % 8; within an XCD the blocks are ordered target, round, token block: an XCD finishes one part of
// one decoder matrix before it touches the next.
struct UnitPlan {
  int ns, ncp, full, rem, q;
  int bf, br;            // blocks per XCD in a full round / in a remainder round
  int64_t tpp;           // tokens per XCD in a remainder round
  int bpx;               // blocks per XCD and target
};

static UnitPlan make_unit_plan(int ns, int ncp, int64_t Tn, int tok_per_block) {
  UnitPlan up;
  up.ns = ns; up.ncp = ncp;
  const int units = ns * ncp;
  up.full = units / 8; up.rem = units % 8;
  up.q = up.rem == 0 ? 1 : (8 % up.rem == 0 ? 8 / up.rem : 8);
  const int rem_rounds = up.rem == 0 ? 0 : (8 % up.rem == 0 ? 1 : up.rem);
  up.tpp = clt_ceil_div(Tn, up.q);
  up.bf = (int)clt_ceil_div(Tn, tok_per_block);
  up.br = (int)clt_ceil_div(up.tpp, tok_per_block);
  up.bpx = up.full * up.bf + rem_rounds * up.br;
  return up;
}

// this block's work: target index (relative), unit -> (slice, column part), its token range and its token block
struct UnitWork { int64_t target; int slice, cpart; int64_t tok_begin, tok_end; int tb; };
__device__ __forceinline__ UnitWork unit_work(const UnitPlan &up, int64_t Tn, int64_t block) {
  UnitWork w;
  const int xcd = (int)(block & 7);
  const int64_t i = block >> 3;
  w.target = i / up.bpx;
  const int j = (int)(i % up.bpx);
  int unit;
  w.tok_begin = 0; w.tok_end = Tn;
  if (j < up.full * up.bf) {
    unit = (j / up.bf) * 8 + xcd; w.tb = j % up.bf;
  } else {
    const int jr = j - up.full * up.bf, rr = jr / up.br;
    w.tb = jr % up.br;
    int tpart;
    if (up.q * up.rem == 8) { unit = up.full * 8 + xcd / up.q; tpart = xcd % up.q; }
    else { unit = up.full * 8 + rr; tpart = xcd; }
    w.tok_begin = (int64_t)tpart * up.tpp;
    w.tok_end = w.tok_begin + up.tpp < Tn ? w.tok_begin + up.tpp : Tn;
  }
  w.cpart = unit % up.ncp; w.slice = unit / up.ncp;
  return w;
}

// ---- one launch per source, or one for all --------------------------------------------------------------
// With a launch per source layer the partial rows [slice][target][token] collect their sources over the launches.  A short
// batch leaves most of the chip idle in every one of them; it gets a single launch over all (source, target) pairs with a
// partial row for each [slice][pair][token], and k_decode_reduce adds a target's sources in the same order: same bits.
// L = 12, d = 768, F = 24576, bf16, 200 per token, us per decode, launch per source / one launch: 1 token 82 / 27,
// 32 tokens 260 / 158, 77 tokens 380 / 310 (780 / 240 on activations whose fullest token has many times the mean: no launch
// waits for it), 256 tokens 730 / 668, 512 tokens 1188 / 1167.
struct PairAt { int src; int64_t t, row; bool first; };      // row: of the partial rows, in units of Tn rows
__device__ __forceinline__ PairAt pair_at(int64_t target, int src, int slice, int64_t L, int64_t t_begin, int64_t t_end,
                                          uint64_t src_mask) {
  PairAt p;
  if (src >= 0) {
    p.src = src; p.t = t_begin + target; p.row = (int64_t)slice * L + p.t;
    p.first = (src_mask & ((1ull << src) - 1ull)) == 0;      // the first source initialises the partial rows
    return p;
  }
  p.src = 0; p.first = true;
  for (;; ++p.src) {
    if (!((src_mask >> p.src) & 1ull)) continue;
    const int64_t from = p.src > t_begin ? p.src : t_begin;
    if (target < t_end - from) { p.t = from + target; break; }
    target -= t_end - from;
  }
  p.row = (int64_t)slice * (L * (L + 1) / 2) + decoder_slot(CLT_TYING_NONE, p.src, p.t, L);
  return p;
}

// ---- quarter-row schedule -------------------------------------------------------------------------
// Large batches, untied or per-source decoders, d a multiple of 256: the feature axis is cut into 2
// slices and the columns into 4 quarters; workgroup b works on part b % 8 = (slice, quarter), so an XCD
// still gathers from one 1/8 of one decoder matrix at a time (F/2 rows x d/4 columns) but a (target,
// token) has 2 partial rows instead of 8: a quarter of the fp32 read-modify-write traffic between source
// launches.  So that a quarter row (384 bytes at d = 768, three whole cache lines) costs no more
// instructions than its share of a whole one, a wavefront fetches FOUR rows per load: each group of
// QLANES = 16 lanes takes one survivor's quarter row, 16 (+8) bytes per lane; every group accumulates
// its own rows and the four groups are added once per token.
constexpr int QLANES = 16;              // lanes per quarter row
constexpr int QROWS = 64 / QLANES;      // rows per load
constexpr int QUARTER_SLICES = 2;       // feature slices; 8 / QUARTER_SLICES column parts
constexpr int QUARTER_PARTS = 8 / QUARTER_SLICES;
template <typename T, int HQ, int HTAIL, int UU, bool PACK> struct PartBatch {
  uint4 wq[UU][HQ > 0 ? HQ : 1];
  uint2 wt8[UU];
  float v[UU];          // !PACK: the activation values
  uint32_t pk[UU];      // PACK: feature index | bf16 value << 16
  // slot QROWS * u + g of the (up to 64) survivors held one per lane goes to lane group g.  Lanes past the
  // end of the list hold feature 0 with value 0: a repeated fetch with weight 0, so nothing is clamped.
  // PACK (bf16, F <= 65536): one cross-lane move per row, and the row offset is a 24-bit multiply-add.
  __device__ __forceinline__ void load(const T *wbase, int64_t d, uint32_t my_pk, int32_t my_col, float my_val, int i0, int n,
                                       int ll, int grp) {
    constexpr int V = WVec<T>::V;
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      const int idx = i0 + QROWS * u + grp;
      if constexpr (PACK) {
        pk[u] = (uint32_t)__builtin_amdgcn_ds_bpermute(idx << 2, (int)my_pk);
        const uint32_t off = __umul24(pk[u] & 0xFFFFu, (uint32_t)d * (uint32_t)sizeof(T)) + (uint32_t)(ll * 16);
        const char *wrow = reinterpret_cast<const char *>(wbase) + off;
#pragma unroll
        for (int c = 0; c < HQ; ++c) wq[u][c] = *reinterpret_cast<const uint4 *>(wrow + c * QLANES * 16);
        if (HTAIL) wt8[u] = *reinterpret_cast<const uint2 *>(wrow + HQ * QLANES * 16 - ll * 8);
      } else {
        const int ci = idx < n ? idx : n - 1;                 // clamp: a repeated fetch, weight 0
        const int32_t f = __shfl(my_col, ci);
        const float vv = __shfl(my_val, ci);
        v[u] = idx < n ? vv : 0.0f;
        const T *wrow = wbase + (int64_t)f * d;
#pragma unroll
        for (int c = 0; c < HQ; ++c) wq[u][c] = *reinterpret_cast<const uint4 *>(wrow + c * QLANES * V + ll * V);
        if (HTAIL) wt8[u] = *reinterpret_cast<const uint2 *>(wrow + HQ * QLANES * V + ll * (V / 2));
      }
    }
  }
  __device__ __forceinline__ uint32_t value_pair(int u) const {
    if constexpr (PACK) return __builtin_amdgcn_perm(pk[u + 1], pk[u], 0x07060302u);   // (value u, value u + 1)
    else return raw16_of<T>(v[u]) | (raw16_of<T>(v[u + 1]) << 16);
  }
  __device__ __forceinline__ void consume(float *acc) const {
    constexpr int V = WVec<T>::V;
    if constexpr (sizeof(T) == 2 && (UU % 2) == 0) {
#pragma unroll
      for (int u = 0; u < UU; u += 2) {
        const uint32_t vv = value_pair(u);
#pragma unroll
        for (int c = 0; c < HQ; ++c) WVec<T>::dot16(acc + c * V, wq[u][c], wq[u + 1][c], vv);
        if (HTAIL) WVec<T>::dot8(acc + HQ * V, wt8[u], wt8[u + 1], vv);
      }
    } else {
#pragma unroll
      for (int u = 0; u < UU; ++u) {
#pragma unroll
        for (int c = 0; c < HQ; ++c) WVec<T>::fma16(acc + c * V, wq[u][c], v[u]);
        if (HTAIL) WVec<T>::fma8(acc + HQ * V, wt8[u], v[u]);
      }
    }
  }
};

constexpr int QUARTER_NTOK = 2;     // tokens per wavefront
// 12 accumulators per lane (d = 768): 72 registers, seven wavefronts per SIMD; wider rows are left alone
template <typename T, int HQ, int HTAIL> constexpr int quarter_min_waves() {
  constexpr int V = 16 / (int)sizeof(T);
  return (sizeof(T) == 2 && HQ * V + (HTAIL ? V / 2 : 0) <= 12) ? 7 : 1;   // fp32 at 7 would spill
}

template <typename T, int HQ, int HTAIL, int UU, bool AFFINE, bool PACK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(quarter_min_waves<T, HQ, HTAIL>(), 8))) void k_decode_quarter(
    const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ wp, const T *__restrict__ foff,
    const T *__restrict__ fscale, int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin, uint64_t src_mask,
    const int32_t *__restrict__ sptr, float *__restrict__ partial, int src_arg, int64_t pitch, UnitPlan up, int64_t t_end) {
  constexpr int V = WVec<T>::V;
  constexpr int NACC = HQ * V + (HTAIL ? V / 2 : 0);      // columns per lane: d / 64
  constexpr int NCP = QUARTER_PARTS;
  const int ns = up.ns;
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int ll = lane & (QLANES - 1), grp = lane / QLANES;
  const bool hi = grp != 0;                    // only the first lane group touches the partial row
  const UnitWork uw = unit_work(up, Tn, (int64_t)blockIdx.x);
  const int slice = uw.slice, cpart = uw.cpart;
  const PairAt at = pair_at(uw.target, src_arg, slice, L, t_begin, t_end, src_mask);
  const int src = at.src;
  const int64_t t = at.t;
  const bool first = at.first;
  const int64_t tok_end = uw.tok_end;
  const int64_t tok0 = uw.tok_begin + ((int64_t)uw.tb * nwv + wv) * QUARTER_NTOK;
  if (tok0 >= tok_end) return;
  int32_t mb = 0, me = 0;
  if (lane < QUARTER_NTOK && tok0 + lane < tok_end) {
    const int64_t r = (int64_t)src * Tn + tok0 + lane;
    mb = sptr[r * (ns + 1) + slice];
    me = sptr[r * (ns + 1) + slice + 1];
  }
  const T *wbase = wp + decoder_slot(tying, src, t, L) * F * pitch + (int64_t)cpart * (d / NCP);
  int32_t nb = __builtin_amdgcn_readlane(mb, 0), ne = __builtin_amdgcn_readlane(me, 0);
  int32_t nxt_col = 0; T nxt_val = Elem<T>::from_raw(0u);
  if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
#pragma unroll
  for (int i = 0; i < QUARTER_NTOK; ++i) {
    const int32_t b = nb, e = ne;
    const int32_t cur_col = nxt_col; const T cur_val = nxt_val;
    if (i + 1 < QUARTER_NTOK) {
      nb = __builtin_amdgcn_readlane(mb, i + 1); ne = __builtin_amdgcn_readlane(me, i + 1);
      nxt_col = 0; nxt_val = Elem<T>::from_raw(0u);
      if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
    }
    if (tok0 + i >= tok_end) break;
    if (b == e && !first) continue;
    // this lane's columns of the partial row (the first lane group writes it): pieces of V, then the tail
    float *prow = partial + (at.row * Tn + tok0 + i) * d + (int64_t)cpart * (d / NCP);
    float old[NACC], acc[NACC];
#pragma unroll
    for (int j = 0; j < NACC; ++j) { old[j] = 0.0f; acc[j] = 0.0f; }
    for (int32_t j0 = b; j0 < e; j0 += 64) {
      const int n = (e - j0) < 64 ? (e - j0) : 64;
      int32_t my_col = cur_col; float my_val = Elem<T>::to_f32(cur_val);
      if (j0 > b) {   // more than 64 survivors in this slice: fetch the next 64
        my_col = 0; my_val = 0.0f;
        if (lane < n) { my_col = col[j0 + lane]; my_val = Elem<T>::to_f32(val[j0 + lane]); }
      }
      if (AFFINE && my_val != 0.0f) {
        if (foff) my_val = Elem<T>::round(my_val + Elem<T>::to_f32(foff[t * F + my_col]));
        if (fscale) my_val = Elem<T>::round(my_val * Elem<T>::to_f32(fscale[t * F + my_col]));
      }
      // two batches of UU row pairs in flight
      const uint32_t my_pk = PACK ? ((uint32_t)my_col | (raw16_of<T>(my_val) << 16)) : 0u;
      PartBatch<T, HQ, HTAIL, UU, PACK> ra, rb;
      constexpr int R = QROWS;
      ra.load(wbase, pitch, my_pk, my_col, my_val, 0, n, ll, grp);
      for (int i0 = 0; i0 < n; i0 += 2 * R * UU) {
        if (i0 + R * UU < n) rb.load(wbase, pitch, my_pk, my_col, my_val, i0 + R * UU, n, ll, grp);
        ra.consume(acc);
        if (i0 + R * UU < n) {
          if (i0 + 2 * R * UU < n) ra.load(wbase, pitch, my_pk, my_col, my_val, i0 + 2 * R * UU, n, ll, grp);
          rb.consume(acc);
        }
      }
    }
    // The old partial row is asked for only now: held across the gathers it would cost 12 registers and
    // one wavefront per SIMD, and the other wavefronts cover its latency better than an early request.
    if (!first && !hi) {
#pragma unroll
      for (int c = 0; c < HQ; ++c) {
#pragma unroll
        for (int j = 0; j < V; j += 4) {
          const float4 q = ldg_stream4(prow + c * QLANES * V + ll * V + j);
          old[c * V + j] = q.x; old[c * V + j + 1] = q.y; old[c * V + j + 2] = q.z; old[c * V + j + 3] = q.w;
        }
      }
      if (HTAIL) {
        if constexpr (V / 2 == 4) {
          const float4 q = ldg_stream4(prow + HQ * QLANES * V + ll * 4);
          old[HQ * V] = q.x; old[HQ * V + 1] = q.y; old[HQ * V + 2] = q.z; old[HQ * V + 3] = q.w;
        } else {
#pragma unroll
          for (int j = 0; j < V / 2; ++j) old[HQ * V + j] = prow[HQ * QLANES * V + ll * (V / 2) + j];
        }
      }
    }
    // the lane groups hold sums over different survivors: add them, in a fixed order (group 0 ends up
    // with ((g0 + g1) + (g2 + g3)))
#pragma unroll
    for (int j = 0; j < NACC; ++j) {
      const float o16 = __shfl_xor(acc[j], 16);
      acc[j] = (lane & 16) ? o16 + acc[j] : acc[j] + o16;
      const float o32 = __shfl_xor(acc[j], 32);
      acc[j] = (lane & 32) ? o32 + acc[j] : acc[j] + o32;
    }
    if (!hi) {
#pragma unroll
      for (int c = 0; c < HQ; ++c) {
#pragma unroll
        for (int j = 0; j < V; j += 4)
          stg_stream4(prow + c * QLANES * V + ll * V + j,
                      make_float4(old[c * V + j] + acc[c * V + j], old[c * V + j + 1] + acc[c * V + j + 1],
                                  old[c * V + j + 2] + acc[c * V + j + 2], old[c * V + j + 3] + acc[c * V + j + 3]));
      }
      if (HTAIL) {
        if constexpr (V / 2 == 4) {
          stg_stream4(prow + HQ * QLANES * V + ll * 4, make_float4(old[HQ * V] + acc[HQ * V], old[HQ * V + 1] + acc[HQ * V + 1],
                                                               old[HQ * V + 2] + acc[HQ * V + 2], old[HQ * V + 3] + acc[HQ * V + 3]));
        } else {
#pragma unroll
          for (int j = 0; j < V / 2; ++j) prow[HQ * QLANES * V + ll * (V / 2) + j] = old[HQ * V + j] + acc[HQ * V + j];
        }
      }
    }
  }
}

// ---- thin lists --------------------------------------------------------------------------------------
// Few survivors per (source, token) - all layers ranked together, a small k: a decoder row is then used by one or two tokens of
// the batch, so keeping an eighth of a matrix in an L2 gains nothing, while the partial rows that the schedule by sources reads
// and writes for every pair are most of its traffic.  Here a wavefront takes one (target, token) and a quarter of the
// columns over all sources: the token's lists become one list, four quarter rows are fetched per load (as above), the sums
// stay in registers and the output row is written once.  XCD x works on quarter x % 4 of one half of the tokens.
// T = 3000, L = 12, F = 24576, d = 768, bf16, 200 survivors per token over all layers: 0.85 ms, 7.1 TB/s of rows out of the caches
// and HBM (by sources 1.53); bounded by the rows in flight: 93 registers leave five wavefronts per SIMD with 16 quarter rows each.
// Workgroups of 8 wavefronts held to 80 registers spill and take 1.1 ms.
// ThinBatch: 4 UU rows of the (up to 64) survivors held one per lane.  In the last batch of a chunk the places past the
// list's end stay zero, so that a row's infinity meets no weight but its own.
template <typename T, int HQ, int HTAIL, int UU> struct ThinBatch {
  uint4 wq[UU][HQ];
  uint2 wt8[UU];
  float v[UU];
  __device__ __forceinline__ void load(const T *wpart, int64_t pitch, int32_t my_row, float my_val, int i0, int n, int ll, int grp) {
    constexpr int V = WVec<T>::V;
    const bool whole = i0 + QROWS * UU <= n;
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      const int idx = i0 + QROWS * u + grp;
      const T *wrow = wpart + (int64_t)__shfl(my_row, idx) * pitch;
      v[u] = __shfl(my_val, idx);
      if (whole || idx < n) {
#pragma unroll
        for (int c = 0; c < HQ; ++c) wq[u][c] = *reinterpret_cast<const uint4 *>(wrow + c * QLANES * V + ll * V);
        if (HTAIL) wt8[u] = *reinterpret_cast<const uint2 *>(wrow + HQ * QLANES * V + ll * (V / 2));
      } else {
        v[u] = 0.0f;
#pragma unroll
        for (int c = 0; c < HQ; ++c) wq[u][c] = make_uint4(0, 0, 0, 0);
        wt8[u] = make_uint2(0, 0);
      }
    }
  }
  __device__ __forceinline__ void consume(float *acc) const {
    constexpr int V = WVec<T>::V;
    if constexpr (sizeof(T) == 2) {
      static_assert(UU % 2 == 0, "rows are multiplied in pairs");
#pragma unroll
      for (int u = 0; u < UU; u += 2) {
        const uint32_t vv = raw16_of<T>(v[u]) | (raw16_of<T>(v[u + 1]) << 16);
#pragma unroll
        for (int c = 0; c < HQ; ++c) WVec<T>::dot16(acc + c * V, wq[u][c], wq[u + 1][c], vv);
        if (HTAIL) WVec<T>::dot8(acc + HQ * V, wt8[u], wt8[u + 1], vv);
      }
    } else {
#pragma unroll
      for (int u = 0; u < UU; ++u) {
#pragma unroll
        for (int c = 0; c < HQ; ++c) WVec<T>::fma16(acc + c * V, wq[u][c], v[u]);
        if (HTAIL) WVec<T>::fma8(acc + HQ * V, wt8[u], v[u]);
      }
    }
  }
};

// The lists of a token over sources 0 .. t as one, a source per lane: where source `lane`'s list begins, less what comes before it
// in the one list, and where it ends there.
struct ThinList {
  int32_t at, end, total;
  __device__ __forceinline__ ThinList(const int32_t *row_ptr, int64_t Tn, int64_t tok, int64_t t, uint64_t src_mask, int lane) {
    at = end = 0;
    if (lane <= t && ((src_mask >> lane) & 1ull)) {
      at = row_ptr[lane * Tn + tok];
      end = row_ptr[lane * Tn + tok + 1] - at;
    }
    at += end;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t up = __shfl_up(end, o);
      if (lane >= o) end += up;
    }
    at -= end;
    total = __builtin_amdgcn_readlane(end, 63);
  }
  // the i-th entry's decoder row and value; beyond the end row 0 and a zero
  template <typename T>
  __device__ __forceinline__ void fetch(int32_t i, const int32_t *col, const T *val, int64_t t, int64_t F, int64_t L, int tying,
                                        int32_t &row, T &v) const {
    row = 0; v = Elem<T>::from_raw(0u);
    int s = 0;
    for (int u = 0; u < (int)t; ++u) s += i >= __builtin_amdgcn_readlane(end, u) ? 1 : 0;
    const int32_t j = __shfl(at, s) + i;
    if (i < total) {
      row = (int32_t)decoder_slot(tying, s, t, L) * (int32_t)F + col[j];
      v = val[j];
    }
  }
};

// A token with a list of more than THIN_LONG (batch-wide top-k gives some tokens many times the average) is left to the end, when
// the workgroup's wavefronts share its chunks of 64 and add their sums in LDS: 25 ns per entry.  One with more than THIN_MOST
// (an outlying token may hold a tenth of all survivors) would keep four workgroups busy long after the others: it goes to
// k_decode_thin_longest.
constexpr int THIN_WAVES = 4, THIN_LONG = 256, THIN_MOST = 8192, THIN_PARTS = 16;

// The longest lists: a workgroup for every target, 128-byte line of the rows and sixteenth of the tokens, in which it looks for
// such lists and sums its columns of them.  A compute unit has some 64 lines on their way, and here an entry is one line, on
// d / 64 (16 bits) as many units: 8 ns per entry.  Usually it finds none: 4 to 8 us.
// us of the decode, L = 6, T = 1500, F = 16384, d = 1024, bf16, 200 per token over all layers, tokens with 0 / 1 x 20 000 / 1 x
// 98 304 / 4 x 50 000 of the 300 000 entries: 260 / 470 / 886 / 478; left to the tokens' own workgroups 256 / 525 / 1909 / 1007;
// the schedule by sources 334 / 412 / 824 / 589.  (In the first workgroups of k_decode_thin's launch it would end with the others, but their
// code together spills: 830 against 795 us for the 3000 tokens above.)
template <typename T>
__global__ __launch_bounds__(THIN_WAVES * 64) void k_decode_thin_longest(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ wp,
    const float *__restrict__ bias_sum, const float *__restrict__ skip_add, void *__restrict__ out, int64_t Tn, int64_t d,
    int64_t F, int64_t L, int tying, int64_t t_end, uint64_t src_mask, int out_f32, int64_t pitch, int units, int64_t max_entries) {
  constexpr int V = WVec<T>::V, COLS = 8 * V, NU = 4;     // 8 lanes per line, 8 rows per load
  if (max_entries >= 0 && row_ptr[L * Tn] > max_entries) return;
  __shared__ int32_t found[THIN_WAVES * 64], n_found[THIN_WAVES];
  __shared__ float shares[THIN_WAVES][COLS];
  const int tid = threadIdx.x, lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ll = lane & 7, grp = lane >> 3;
  // (the workgroups of one part of the tokens follow each other, over all XCDs)
  const int per_part = gridDim.x / THIN_PARTS, part = blockIdx.x / per_part, of_part = blockIdx.x - part * per_part, unit = of_part % units;
  const int64_t t = t_end - 1 - of_part / units, begin = Tn * part / THIN_PARTS, end = Tn * (part + 1) / THIN_PARTS;
  const T *wpart = wp + (int64_t)unit * COLS + ll * V;
  for (int64_t tok0 = begin; tok0 < end; tok0 += THIN_WAVES * 64) {
    const int64_t mine = tok0 + tid;
    int32_t n = 0;
    if (mine < end) {
      for (int s0 = 0; s0 <= (int)t; s0 += 8) {            // eight sources asked for at once
        int32_t a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int32_t *p = row_ptr + (s0 + u <= (int)t ? s0 + u : 0) * Tn + mine;
          a[u] = p[0]; b[u] = p[1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (s0 + u <= (int)t && ((src_mask >> (s0 + u)) & 1ull)) n += b[u] - a[u];
      }
    }
    const uint64_t votes = __ballot(n > THIN_MOST);
    if (lane == 0) n_found[wv] = __popcll(votes);
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < THIN_WAVES; ++w) {
      before += w < wv ? n_found[w] : 0;
      all += n_found[w];
    }
    if (n > THIN_MOST) found[before + __builtin_amdgcn_mbcnt_hi((uint32_t)(votes >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)votes, 0u))] = tid;
    __syncthreads();
    for (int k = 0; k < all; ++k) {
      const int64_t tok = tok0 + found[k];
      const ThinList list(row_ptr, Tn, tok, t, src_mask, lane);
      float acc[V];
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] = 0.0f;
      int32_t row, next_row;
      T v, next_v;
      list.fetch(wv * 64 + lane, col, val, t, F, L, tying, row, v);
      for (int32_t j0 = wv * 64; j0 < list.total; j0 += THIN_WAVES * 64) {
#pragma unroll 1
        for (int h = 0; h < 8; h += NU) {
          uint4 w[NU];
          float a[NU];
#pragma unroll
          for (int u = 0; u < NU; ++u) {                   // past the end: zeros times zeros
            const int idx = 8 * (h + u) + grp;
            a[u] = __shfl(Elem<T>::to_f32(v), idx);
            const int64_t at = (int64_t)__shfl(row, idx) * pitch;
            w[u] = make_uint4(0, 0, 0, 0);
            if (j0 + idx < list.total) w[u] = *reinterpret_cast<const uint4 *>(wpart + at);
          }
          if (h == 0) list.fetch(j0 + THIN_WAVES * 64 + lane, col, val, t, F, L, tying, next_row, next_v);
#pragma unroll
          for (int u = 0; u < NU; u += 2) {
            if constexpr (sizeof(T) == 2) WVec<T>::dot16(acc, w[u], w[u + 1], raw16_of<T>(a[u]) | (raw16_of<T>(a[u + 1]) << 16));
            else {
              WVec<T>::fma16(acc, w[u], a[u]);
              WVec<T>::fma16(acc, w[u + 1], a[u + 1]);
            }
          }
        }
        row = next_row; v = next_v;
      }
#pragma unroll
      for (int j = 0; j < V; ++j) {
        acc[j] += __shfl_xor(acc[j], 8);
        acc[j] += __shfl_xor(acc[j], 16);
        acc[j] += __shfl_xor(acc[j], 32);
        if (grp == 0) shares[wv][ll * V + j] = acc[j];
      }
      __syncthreads();
      if (tid < COLS) {
        float y = (shares[0][tid] + shares[1][tid]) + (shares[2][tid] + shares[3][tid]);
        const int64_t c = (int64_t)unit * COLS + tid, at = (t * Tn + tok) * d + c;
        if (bias_sum) y += bias_sum[t * d + c];
        if (skip_add) y += skip_add[at];
        if (out_f32 || sizeof(T) == 4) ((float *)out)[at] = y;
        else ((T *)out)[at] = Elem<T>::from_f32(y);
      }
      __syncthreads();
    }
  }
}

template <typename T, int HQ, int HTAIL>
__global__ __launch_bounds__(THIN_WAVES * 64) void k_decode_thin(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ wp,
    const float *__restrict__ bias_sum, const float *__restrict__ skip_add, void *__restrict__ out, int64_t Tn, int64_t d,
    int64_t F, int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int out_f32, int64_t pitch, int64_t max_entries) {
  constexpr int V = WVec<T>::V, UU = 2, R = QROWS * UU;
  if (max_entries >= 0 && row_ptr[L * Tn] > max_entries) return;
  constexpr int NACC = HQ * V + (HTAIL ? V / 2 : 0);      // columns per lane: d / 64
  __shared__ int32_t totals[THIN_WAVES];
  __shared__ float shares[THIN_WAVES][NACC][QLANES];
  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ll = lane & (QLANES - 1), grp = lane / QLANES;
  const int cpart = (int)(blockIdx.x & 3), half = (int)((blockIdx.x >> 2) & 1);
  const int64_t idx = blockIdx.x >> 3, in_half = (Tn + 1) / 2, per_t = (in_half + THIN_WAVES - 1) / THIN_WAVES;
  const int64_t t = t_end - 1 - idx / per_t;               // longest first
  const int64_t in0 = (idx % per_t) * THIN_WAVES;          // of the half: the first wavefront's token
  const T *wpart = wp + (int64_t)cpart * (d / 4);

  struct Entry { int32_t row; T v; };
  float acc[NACC];
  // every `step`-th chunk of the token's list from chunk `from` on; the lane groups' sums end up as ((g0 + g1) + (g2 + g3))
  auto gather = [&](const ThinList &list, int from, int step) {
#pragma unroll
    for (int j = 0; j < NACC; ++j) acc[j] = 0.0f;
    Entry next;
    list.fetch(from * 64 + lane, col, val, t, F, L, tying, next.row, next.v);
    for (int32_t j0 = from * 64; j0 < list.total; j0 += step * 64) {
      const int32_t my_row = next.row;
      const float my_val = Elem<T>::to_f32(next.v);
      const int n = list.total - j0 < 64 ? list.total - j0 : 64;
      ThinBatch<T, HQ, HTAIL, UU> ra, rb;
      ra.load(wpart, pitch, my_row, my_val, 0, n, ll, grp);
      if (j0 + step * 64 < list.total) list.fetch(j0 + step * 64 + lane, col, val, t, F, L, tying, next.row, next.v);
      for (int i0 = 0; i0 < n; i0 += 2 * R) {
        if (i0 + R < n) rb.load(wpart, pitch, my_row, my_val, i0 + R, n, ll, grp);
        ra.consume(acc);
        if (i0 + R < n) {
          if (i0 + 2 * R < n) ra.load(wpart, pitch, my_row, my_val, i0 + 2 * R, n, ll, grp);
          rb.consume(acc);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NACC; ++j) {
      acc[j] += __shfl_xor(acc[j], 16);
      acc[j] += __shfl_xor(acc[j], 32);
    }
  };
  auto emit = [&](int64_t tok) {
    if (grp != 0) return;
    const int64_t col0 = (int64_t)cpart * (d / 4), at = (t * Tn + tok) * d;
    auto emit4 = [&](int64_t o, const float *a) {
      float4 y = make_float4(a[0], a[1], a[2], a[3]);
      if (bias_sum) { const float4 b = *reinterpret_cast<const float4 *>(bias_sum + t * d + o); y.x += b.x; y.y += b.y; y.z += b.z; y.w += b.w; }
      if (skip_add) { const float4 b = *reinterpret_cast<const float4 *>(skip_add + at + o); y.x += b.x; y.y += b.y; y.z += b.z; y.w += b.w; }
      if (out_f32 || sizeof(T) == 4) *reinterpret_cast<float4 *>((float *)out + at + o) = y;
      else *reinterpret_cast<uint2 *>((uint16_t *)out + at + o) = make_uint2(pack_pair<T>(y.x, y.y), pack_pair<T>(y.z, y.w));
    };
#pragma unroll
    for (int c = 0; c < HQ; ++c)
#pragma unroll
      for (int j = 0; j < V; j += 4) emit4(col0 + c * QLANES * V + ll * V + j, acc + c * V + j);
    if constexpr (HTAIL && V == 8) emit4(col0 + HQ * QLANES * V + ll * 4, acc + HQ * V);
  };

  // w < 0: each wavefront its own token; w >= 0: all of them wavefront w's, if that was left (one instance of the loop for both)
  for (int w = -1; w < THIN_WAVES; ++w) {
    if (w == 0) __syncthreads();
    const int64_t in = in0 + (w < 0 ? wv : w), tok = half * in_half + in;
    const bool on = in < in_half && tok < Tn;
    if (w >= 0 && (totals[w] <= THIN_LONG || totals[w] > THIN_MOST)) continue;     // the same for the whole workgroup
    const ThinList list(row_ptr, Tn, on ? tok : 0, t, on ? src_mask : 0ull, lane);
    if (w < 0) {
      if (lane == 0) totals[wv] = list.total;
      if (!on || list.total > THIN_LONG) continue;
    }
    gather(list, w < 0 ? 0 : wv, w < 0 ? 1 : THIN_WAVES);
    if (w >= 0) {
      if (grp == 0) {
#pragma unroll
        for (int j = 0; j < NACC; ++j) shares[wv][j][ll] = acc[j];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NACC; ++j) {
        acc[j] = 0.0f;
#pragma unroll
        for (int o = 0; o < THIN_WAVES; o += 2) acc[j] += shares[o][j][ll] + shares[o + 1][j][ll];
      }
      __syncthreads();
    }
    if (w < 0 || wv == w) emit(tok);
  }
}

// ---- line schedule ---------------------------------------------------------------------------------
// Large batches, untied or per-source decoders, rows that are whole 128-byte cache lines: the COLUMNS are
// cut into parts of exactly one cache line (64 bf16 / 32 fp32), so the piece of a decoder matrix that an
// XCD gathers from while all tokens stream past is F x 128 bytes (3.0 MiB at F = 24576, inside its 4 MiB
// L2; wider feature axes are cut into `ns` slices to stay there).  The units of work (slice, column part,
// token part) are dealt to the XCDs in rounds - unit u runs on XCD u % 8 in round u / 8 - and the token
// axis is cut into `ntp` parts only to make their number a multiple of 8.  A load instruction fetches the
// line of EIGHT survivors (8 lanes x 16 bytes each); every lane group accumulates its own survivors and a
// butterfly that halves the accumulators at every step (reduce-scatter: 7 shuffles for 8 accumulators)
// leaves each lane with the finished sum of one column.  With ns = 1 a (target, token) has one fp32
// partial row, read and written once per source layer.
constexpr int LINE_UU = 2;                // loads per batch (two batches in flight)
constexpr int64_t LINE_L2_BYTES = 3407872;   // 3.25 MiB: the part of a matrix one XCD works on stays below this

template <typename T, int UU, bool PACK> struct LineBatch {
  uint4 wq[UU];
  float v[UU];          // !PACK: the activation values
  uint32_t pk[UU];      // PACK: feature index | bf16 value << 16
  // entry 8 * u + grp of the (up to 64) survivors held one per lane goes to lane group grp; lanes past the
  // end of the list hold feature 0 with value 0 (a repeated fetch, weight 0)
  __device__ __forceinline__ void load(const T *wbase, int64_t rstride, uint32_t my_pk, int32_t my_col, float my_val, int i0,
                                       int n, int ll, int grp) {
    constexpr int V = WVec<T>::V;
#pragma unroll
    for (int u = 0; u < UU; ++u) {
      const int idx = i0 + 8 * u + grp;
      if constexpr (PACK) {
        pk[u] = (uint32_t)__builtin_amdgcn_ds_bpermute(idx << 2, (int)my_pk);
        const uint32_t off = __umul24(pk[u] & 0xFFFFu, (uint32_t)rstride * (uint32_t)sizeof(T)) + (uint32_t)(ll * 16);
        wq[u] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(wbase) + off);
      } else {
        const int ci = idx < n ? idx : n - 1;
        const int32_t f = __shfl(my_col, ci);
        const float vv = __shfl(my_val, ci);
        v[u] = idx < n ? vv : 0.0f;
        wq[u] = *reinterpret_cast<const uint4 *>(wbase + (int64_t)f * rstride + ll * V);
      }
    }
  }
  __device__ __forceinline__ void consume(float *acc) const {
    if constexpr (sizeof(T) == 2 && (UU % 2) == 0) {
#pragma unroll
      for (int u = 0; u < UU; u += 2) {
        uint32_t vb;
        if constexpr (PACK) vb = __builtin_amdgcn_perm(pk[u + 1], pk[u], 0x07060302u);
        else vb = raw16_of<T>(v[u]) | (raw16_of<T>(v[u + 1]) << 16);
        WVec<T>::dot16(acc, wq[u], wq[u + 1], vb);
      }
    } else {
#pragma unroll
      for (int u = 0; u < UU; ++u) WVec<T>::fma16(acc, wq[u], v[u]);
    }
  }
};

// the n <= 64 survivors that a wavefront holds one per lane, two batches of loads in flight
template <typename T, bool PACK>
__device__ __forceinline__ void line_chunk(float *acc, const T *wbase, int64_t pitch, int32_t my_col, float my_val, int n, int ll, int grp) {
  // 16 bits: feature index (< 65536) and value travel to their lane group in one 32-bit word
  const uint32_t my_pk = PACK ? ((uint32_t)my_col | (raw16_of<T>(my_val) << 16)) : 0u;
  constexpr int R = 8 * LINE_UU;                 // survivors per batch
  LineBatch<T, LINE_UU, PACK> ra, rb;
  ra.load(wbase, pitch, my_pk, my_col, my_val, 0, n, ll, grp);
  for (int i0 = 0; i0 < n; i0 += 2 * R) {
    if (i0 + R < n) rb.load(wbase, pitch, my_pk, my_col, my_val, i0 + R, n, ll, grp);
    ra.consume(acc);
    if (i0 + R < n) {
      if (i0 + 2 * R < n) ra.load(wbase, pitch, my_pk, my_col, my_val, i0 + 2 * R, n, ll, grp);
      rb.consume(acc);
    }
  }
}

// Reduce-scatter of 8 sums over the eight lane groups (fixed order): every step hands half of the accumulators to the partner
// group and adds the half that comes back, so a lane ends with the sum of ONE column, 8 * (lane % 8) + lane / 8.
__device__ __forceinline__ float line_scatter8(const float *acc, int grp) {
  float a4[4], a2[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float keep = (grp & 4) ? acc[j + 4] : acc[j], send = (grp & 4) ? acc[j] : acc[j + 4];
    a4[j] = keep + __shfl_xor(send, 32);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float keep = (grp & 2) ? a4[j + 2] : a4[j], send = (grp & 2) ? a4[j] : a4[j + 2];
    a2[j] = keep + __shfl_xor(send, 16);
  }
  const float keep = (grp & 1) ? a2[1] : a2[0], send = (grp & 1) ? a2[0] : a2[1];
  return keep + __shfl_xor(send, 8);
}

template <typename T, bool AFFINE, bool PACK, int NTOK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_decode_line(
    const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ wp, const T *__restrict__ foff,
    const T *__restrict__ fscale, int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin, uint64_t src_mask,
    const int32_t *__restrict__ sptr, float *__restrict__ partial, int src_arg, UnitPlan lp, int64_t pitch, int64_t t_end) {
  constexpr int V = WVec<T>::V;                     // elements per lane: 16 bytes
  constexpr int LW = 8 * V;                         // columns per part: one 128-byte line
  constexpr int LINE_NTOK = NTOK;
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int ll = lane & 7, grp = lane >> 3;
  const int ns = lp.ns;
  const UnitWork uw = unit_work(lp, Tn, (int64_t)blockIdx.x);
  const int cpart = uw.cpart, slice = uw.slice;
  const PairAt at = pair_at(uw.target, src_arg, slice, L, t_begin, t_end, src_mask);
  const int src = at.src;
  const int64_t t = at.t;
  const bool first = at.first;
  const int64_t part_end = uw.tok_end;
  const int64_t tok0 = uw.tok_begin + ((int64_t)uw.tb * nwv + wv) * LINE_NTOK;
  if (tok0 >= part_end) return;
  int32_t mb = 0, me = 0;
  if (lane < LINE_NTOK && tok0 + lane < part_end) {
    const int64_t r = (int64_t)src * Tn + tok0 + lane;
    mb = sptr[r * (ns + 1) + slice];
    me = sptr[r * (ns + 1) + slice + 1];
  }
  const T *wbase = wp + decoder_slot(tying, src, t, L) * F * pitch + (int64_t)cpart * LW;
  int32_t nb = __builtin_amdgcn_readlane(mb, 0), ne = __builtin_amdgcn_readlane(me, 0);
  int32_t nxt_col = 0; T nxt_val = Elem<T>::from_raw(0u);
  if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
#pragma unroll
  for (int it = 0; it < LINE_NTOK; ++it) {
    const int32_t b = nb, e = ne;
    const int32_t cur_col = nxt_col; const T cur_val = nxt_val;
    if (it + 1 < LINE_NTOK) {
      nb = __builtin_amdgcn_readlane(mb, it + 1); ne = __builtin_amdgcn_readlane(me, it + 1);
      nxt_col = 0; nxt_val = Elem<T>::from_raw(0u);
      if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
    }
    if (tok0 + it >= part_end) break;
    if (b == e && !first) continue;
    float acc[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = 0.0f;
    for (int32_t j0 = b; j0 < e; j0 += 64) {
      const int n = (e - j0) < 64 ? (e - j0) : 64;
      int32_t my_col = cur_col; float my_val = Elem<T>::to_f32(cur_val);
      if (j0 > b) {   // more than 64 survivors in this slice: fetch the next 64
        my_col = 0; my_val = 0.0f;
        if (lane < n) { my_col = col[j0 + lane]; my_val = Elem<T>::to_f32(val[j0 + lane]); }
      }
      if (AFFINE && my_val != 0.0f) {
        if (foff) my_val = Elem<T>::round(my_val + Elem<T>::to_f32(foff[t * F + my_col]));
        if (fscale) my_val = Elem<T>::round(my_val * Elem<T>::to_f32(fscale[t * F + my_col]));
      }
      line_chunk<T, PACK>(acc, wbase, pitch, my_col, my_val, n, ll, grp);
    }
    // reduce-scatter over the eight lane groups (fixed order): a lane ends with the sum of ONE column
    float r; int csel; bool writer = true;
    if constexpr (V == 8) {
      r = line_scatter8(acc, grp);
      csel = ll * 8 + grp;
    } else {
      float a2[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float keep = (grp & 4) ? acc[j + 2] : acc[j], send = (grp & 4) ? acc[j] : acc[j + 2];
        a2[j] = keep + __shfl_xor(send, 32);
      }
      const float keep = (grp & 2) ? a2[1] : a2[0], send = (grp & 2) ? a2[0] : a2[1];
      const float a1 = keep + __shfl_xor(send, 16);
      const float o = __shfl_xor(a1, 8);
      r = (grp & 1) ? o + a1 : a1 + o;             // both lanes of a pair form the same sum
      csel = ll * 4 + ((grp >> 2) & 1) * 2 + ((grp >> 1) & 1);
      writer = (grp & 1) == 0;
    }
    float *pp = partial + (at.row * Tn + tok0 + it) * d + (int64_t)cpart * LW + csel;
    if (writer) {
      const float old = first ? 0.0f : __builtin_nontemporal_load(pp);
      __builtin_nontemporal_store(old + r, pp);
    }
  }
}

// A list that is longer than `only_above`, in one launch and without a workspace; nothing happens to a shorter one.  For the
// threshold list that outgrew what the tiles were given: the host does not know, so the launch is always made, and its
// OVER_BLOCKS workgroups - as many as are resident, taking the plan's blocks in turn - leave at once in the ordinary case.
//
// Units of one cache line of columns as in the line schedule, with every source in the place of one: a workgroup keeps the sums
// of up to OVER_TOKENS tokens in LDS and takes one source after the other over all of them, so that the workgroups of an XCD
// gather from about one matrix at a time, which its L2 holds.  Bound by that gather, as the schedules with a launch per source
// are, whose partial rows it does without.  Those / this, ms, bf16, untied, 200 survivors per token: L = 12, d = 768, F = 24576,
// 4096 tokens 5.90 / 6.05, 512 tokens 1.15 / 1.07; L = 24, d = 1024, F = 32768 (a line of every row is more than an L2), 2048
// tokens 17.2 / 20.4; 50 per token: L = 4, F = 8192, 512 tokens, d = 2560 0.159 / 0.161, d = 4096 0.245 / 0.245.  Hence
// also how many tokens a workgroup takes: a 64th, so that the workgroups of an XCD share one unit (a 288-token share, with
// four units of the XCD in flight: 10.2 ms in place of 6.05).
// Measured and dropped: the sums of two tokens at a time in registers over all sources (13.2 ms: the wavefronts of an XCD
// drift apart over the sources, and no L2 holds them all); one pass of k_decode (11.4 ms, 32.3, and 4.2 and 6.7 ms of the
// last two, whose rows only k_decode_generic takes).
constexpr int OVER_WAVES = 16, OVER_TOKENS = 288, OVER_BLOCKS = 2 * 256;
template <typename T, bool PACK>
__global__ __launch_bounds__(OVER_WAVES * 64) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_decode_over(
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ wp,
    const float *__restrict__ bias_sum, const float *__restrict__ skip_add, void *__restrict__ out, int64_t Tn, int64_t d, int64_t F,
    int64_t L, int tying, int t_end, uint64_t src_mask, int out_f32, UnitPlan lp, int ntok, int64_t pitch, int64_t blocks,
    int64_t only_above) {
  extern __shared__ float sums[];                            // [ntok][64]
  if (row_ptr[L * Tn] <= only_above) return;
  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ll = lane & 7, grp = lane >> 3;
  for (int64_t block = blockIdx.x; block < blocks; block += gridDim.x) {
    const UnitWork uw = unit_work(lp, Tn, block);
    const int t = t_end - 1 - (int)uw.target;                // longest first
    const int64_t tok0 = uw.tok_begin + (int64_t)uw.tb * ntok + wv;      // this wavefront's: every OVER_WAVES-th from here
    const int64_t left = (uw.tok_end < tok0 - wv + ntok ? uw.tok_end : tok0 - wv + ntok) - tok0;
    const int n_mine = left > 0 ? (int)((left + OVER_WAVES - 1) / OVER_WAVES) : 0;
    float *mine = sums + wv * 64;
    for (int i = 0; i < n_mine; ++i) mine[i * (OVER_WAVES * 64) + lane] = 0.0f;
    for (uint64_t m = src_mask & ((2ull << t) - 1ull); m != 0; m &= m - 1) {
      const int s = __ffsll((unsigned long long)m) - 1;
      __syncthreads();                                       // the workgroup stays together
      const T *wbase = wp + decoder_slot(tying, s, t, L) * F * pitch + (int64_t)uw.cpart * 64;
      int32_t mb = 0, me = 0;                                // the tokens' lists, a lane each
      if (lane < n_mine) {
        const int64_t r = (int64_t)s * Tn + tok0 + lane * OVER_WAVES;
        mb = row_ptr[r]; me = row_ptr[r + 1];
      }
      int32_t nb = __builtin_amdgcn_readlane(mb, 0), ne = __builtin_amdgcn_readlane(me, 0), nxt_col = 0;
      T nxt_val = Elem<T>::from_raw(0u);
      if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
      for (int i = 0; i < n_mine; ++i) {
        const int32_t b = nb, e = ne, cur_col = nxt_col;
        const T cur_val = nxt_val;
        if (i + 1 < n_mine) {
          nb = __builtin_amdgcn_readlane(mb, i + 1); ne = __builtin_amdgcn_readlane(me, i + 1);
          nxt_col = 0; nxt_val = Elem<T>::from_raw(0u);
          if (lane < ne - nb) { nxt_col = col[nb + lane]; nxt_val = val[nb + lane]; }
        }
        if (b == e) continue;
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int32_t j0 = b; j0 < e; j0 += 64) {
          const int n = (e - j0) < 64 ? (e - j0) : 64;
          int32_t my_col = cur_col; float my_val = Elem<T>::to_f32(cur_val);
          if (j0 > b) {
            my_col = 0; my_val = 0.0f;
            if (lane < n) { my_col = col[j0 + lane]; my_val = Elem<T>::to_f32(val[j0 + lane]); }
          }
          line_chunk<T, PACK>(acc, wbase, pitch, my_col, my_val, n, ll, grp);
        }
        mine[i * (OVER_WAVES * 64) + ll * 8 + grp] += line_scatter8(acc, grp);
      }
    }
    for (int i = 0; i < n_mine; ++i) {
      const int64_t o = (int64_t)uw.cpart * 64 + ll * 8 + grp, at = ((int64_t)t * Tn + tok0 + i * OVER_WAVES) * d + o;
      float y = mine[i * (OVER_WAVES * 64) + ll * 8 + grp];
      if (bias_sum) y += bias_sum[(int64_t)t * d + o];
      if (skip_add) y += skip_add[at];
      if (out_f32) ((float *)out)[at] = y;
      else ((T *)out)[at] = Elem<T>::from_f32(y);
    }
  }
}

// sptr[r][j] = first survivor of row r whose feature index is >= j * F / ns  (j = 0..ns)
__global__ void k_slice_ptr(const int32_t *row_ptr, const int32_t *col, int64_t R, int64_t F, int ns, int32_t *sptr) {
  const int64_t total = R * (ns + 1);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / (ns + 1);
    const int j = (int)(i - r * (ns + 1));
    const int32_t bound = (int32_t)(((int64_t)j * F) / ns);
    int32_t lo = row_ptr[r], hi = row_ptr[r + 1];
    while (lo < hi) {
      int32_t mid = lo + ((hi - lo) >> 1);
      if (col[mid] < bound) lo = mid + 1; else hi = mid;
    }
    sptr[i] = lo;
  }
}

// out[t][tok][:] = sum over slices (fixed order) + bias + skip, rounded once.  4 elements per thread.
template <typename T>
__global__ void k_decode_reduce(const float *__restrict__ partial, const float *__restrict__ bias_sum,
                                const float *__restrict__ skip_add, void *__restrict__ out, int64_t Tn, int64_t d,
                                int64_t L, int64_t t_begin, int64_t t_end, int ns, int out_f32, uint64_t src_mask,
                                bool pairs = false) {
  const int64_t per_t = Tn * d, span = (t_end - t_begin) * per_t, slice_stride = L * per_t;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < span; i += (int64_t)gridDim.x * blockDim.x * 4) {
    const int64_t g = t_begin * per_t + i;          // index into [L][T][d]
    const int64_t t = g / per_t, o = g % d;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pairs) {                                      // a partial row per (source, target): sources first, then slices
      const int64_t np = L * (L + 1) / 2, at = g - t * per_t;
      for (int sl = 0; sl < ns; ++sl) {
        float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (int64_t s = 0; s <= t; ++s) {
          if (!((src_mask >> s) & 1ull)) continue;
          const float4 q = *reinterpret_cast<const float4 *>(partial + (sl * np + decoder_slot(CLT_TYING_NONE, s, t, L)) * per_t + at);
          b.x += q.x; b.y += q.y; b.z += q.z; b.w += q.w;
        }
        if (sl == 0) a = b;
        else { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
      }
    } else if (src_mask & ((2ull << t) - 1ull)) {     // some source <= t wrote partial rows
      a = *reinterpret_cast<const float4 *>(partial + g);
      for (int sl = 1; sl < ns; ++sl) {
        float4 b = *reinterpret_cast<const float4 *>(partial + sl * slice_stride + g);
        a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
      }
    }
    if (bias_sum) { a.x += bias_sum[t * d + o]; a.y += bias_sum[t * d + o + 1]; a.z += bias_sum[t * d + o + 2]; a.w += bias_sum[t * d + o + 3]; }
    if (skip_add) { float4 k = *reinterpret_cast<const float4 *>(skip_add + g); a.x += k.x; a.y += k.y; a.z += k.z; a.w += k.w; }
    if (out_f32) *reinterpret_cast<float4 *>((float *)out + g) = a;
    else if (sizeof(T) == 4) *reinterpret_cast<float4 *>((float *)out + g) = a;
    else {
      uint2 o2;
      o2.x = pack_pair<T>(a.x, a.y);
      o2.y = pack_pair<T>(a.z, a.w);
      *reinterpret_cast<uint2 *>((bf16_t *)out + g) = o2;
    }
  }
}

// Any d (no alignment assumption): lanes stride over the output row one element at a time.
template <typename T>
__global__ __launch_bounds__(256) void k_decode_generic(
    const int32_t *row_ptr, const int32_t *col, const T *val, const T *wp, const float *bias_sum,
    const T *foff, const T *fscale, const float *skip_add, void *out, int64_t Tn, int64_t d,
    int64_t F, int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int out_f32, int64_t pitch) {
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int64_t blocks_per_t = (Tn + nwv - 1) / nwv;
  const int64_t t = t_end - 1 - (int64_t)blockIdx.x / blocks_per_t;
  const int64_t tok = ((int64_t)blockIdx.x % blocks_per_t) * nwv + wv;
  if (tok >= Tn) return;
  for (int64_t o0 = 0; o0 < d; o0 += 64) {
    const int64_t o = o0 + lane;
    float acc = 0.0f;
    for (int64_t s = 0; s <= t; ++s) {
      if (!((src_mask >> s) & 1ull)) continue;
      const int64_t r = s * Tn + tok;
      const T *wbase = wp + decoder_slot(tying, s, t, L) * F * pitch;
      for (int32_t j = row_ptr[r]; j < row_ptr[r + 1]; ++j) {
        const int32_t f = col[j];
        float v = Elem<T>::to_f32(val[j]);
        if (v != 0.0f) {
          if (foff) v = Elem<T>::round(v + Elem<T>::to_f32(foff[t * F + f]));
          if (fscale) v = Elem<T>::round(v * Elem<T>::to_f32(fscale[t * F + f]));
        }
        if (o < d) acc = fmaf(v, Elem<T>::to_f32(wbase[(int64_t)f * pitch + o]), acc);
      }
    }
    if (o < d) {
      if (bias_sum) acc += bias_sum[t * d + o];
      if (skip_add) acc += skip_add[(t * Tn + tok) * d + o];
      if (out_f32) ((float *)out)[(t * Tn + tok) * d + o] = acc;
      else ((T *)out)[(t * Tn + tok) * d + o] = Elem<T>::from_f32(acc);
    }
  }
}

// [d][F] -> [F][d] through a 64x64 LDS tile (coalesced on both sides).
template <typename T>
__global__ __launch_bounds__(256) void k_pack(const T *src, T *dst, int64_t d, int64_t F,
                                              int64_t in_stride, int64_t out_stride, int64_t pitch) {
  __shared__ T tile[64][65];
  const T *s = src + (int64_t)blockIdx.z * in_stride;
  T *o = dst + (int64_t)blockIdx.z * out_stride;
  const int64_t f0 = (int64_t)blockIdx.x * 64, d0 = (int64_t)blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    int64_t dd = d0 + i, ff = f0 + tx;
    if (dd < d && ff < F) tile[i][tx] = s[dd * F + ff];
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    int64_t ff = f0 + i, dd = d0 + tx;
    if (ff < F && dd < d) o[ff * pitch + dd] = tile[tx][i];
  }
}

// The same for the matrices whose flag is set, addressed through a table of parameter pointers: FP_PACK_BLOCKS
// workgroups per matrix walk its 64 x 64 tiles; a matrix whose flag is clear costs its workgroups one load.
constexpr int FP_PACK_BLOCKS = 64;
template <typename T>
__global__ __launch_bounds__(256) void k_pack_if(T *const *w_refs, T *dst, int64_t d, int64_t F, int64_t pitch,
                                                 const int32_t *changed) {
  __shared__ T tile[64][65];
  const int z = blockIdx.y;
  if (changed[z] == 0) return;
  const T *s = w_refs[z];
  T *o = dst + (int64_t)z * F * pitch;
  const int64_t tf = (F + 63) / 64, td = (d + 63) / 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int64_t tile_i = blockIdx.x; tile_i < tf * td; tile_i += gridDim.x) {
    const int64_t f0 = (tile_i % tf) * 64, d0 = (tile_i / tf) * 64;
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
      int64_t dd = d0 + i, ff = f0 + tx;
      if (dd < d && ff < F) tile[i][tx] = s[dd * F + ff];
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
      int64_t ff = f0 + i, dd = d0 + tx;
      if (ff < F && dd < d) o[ff * pitch + dd] = tile[tx][i];
    }
  }
}

// Fingerprint of every decoder parameter [d][F]: a sum (order-free, so the workgroups of a matrix add to it with
// atomics) of mixed 32-bit words from sampled runs of 64 words.  A matrix of up to FP_CHUNKS runs is taken whole.
// A larger one gives one run per row, on a diagonal: row r gives run (61 r + r / runs_per_row) mod runs_per_row, so
// every row is looked at and every column in d / runs_per_row rows - a write to a whole row, a whole column or the
// whole matrix cannot be missed, and the sample is d x 256 bytes (0.5 % of a 768 x 24576 matrix).  Rows that are not
// a whole number of words fall back to FP_CHUNKS evenly spread runs.
// FP_BLOCKS workgroups per matrix (a CU keeps only ~64 line requests in flight, so a matrix's rows are spread over
// several CUs).  state holds one 128-byte line per matrix - FP_BLOCKS partial sums, the stored fingerprint and an
// arrival counter - so that the workgroups of different matrices never meet on a cache line; the last workgroup of
// a matrix to arrive adds the partial sums, compares, stores and leaves the counter at zero.
constexpr int FP_BLOCKS = 8;
constexpr int FP_STATE_WORDS = 16;
constexpr int FP_CHUNKS = 4096;
__device__ __forceinline__ unsigned long long fp_mix(uint32_t word, uint32_t index) {
  unsigned long long h = ((unsigned long long)word << 32) | (unsigned long long)(index * 0x9E3779B1u + 0x7F4A7C15u);
  h ^= h >> 29; h *= 0xBF58476D1CE4E5B9ull; h ^= h >> 32; h *= 0x94D049BB133111EBull; h ^= h >> 29;
  return h;
}
__global__ __launch_bounds__(256) void k_fingerprint(const uint32_t *const *w_refs, int64_t words, int64_t rows,
                                                     int64_t words_per_row, unsigned long long *state,
                                                     int32_t *changed, int store_only) {
  __shared__ unsigned long long red[4];
  const int z = blockIdx.y, lane = lane_id(), wv = threadIdx.x >> 6;
  const uint32_t *w = w_refs[z];
  const int64_t n_chunks = (words + 63) / 64;
  const int64_t rpr = words_per_row > 0 ? (words_per_row + 63) / 64 : 0;      // runs per row
  const bool whole = n_chunks <= FP_CHUNKS, diagonal = !whole && rpr > 0;
  const int64_t take = whole ? n_chunks : diagonal ? rows : FP_CHUNKS;
  unsigned long long h = 0;
  // all runs of a wavefront in flight at once (24 of 768 rows): a handful of independent loads per lane, all latency (78 matrices of
  // 768 x 24576, bf16: 30 -> 24 us; 300 of 1024 x 32768 170 -> 147)
  constexpr int FP_UNROLL = 24;
  const int64_t step = (int64_t)FP_BLOCKS * 4;
  for (int64_t j0 = (int64_t)blockIdx.x * 4 + wv; j0 < take; j0 += step * FP_UNROLL) {
    uint32_t v[FP_UNROLL];
    int64_t at[FP_UNROLL];
#pragma unroll
    for (int u = 0; u < FP_UNROLL; ++u) {
      const int64_t j = j0 + u * step;
      int64_t i = -1;
      if (j < take) {
        if (whole) i = j * 64 + lane;
        else if (diagonal) {
          const uint32_t r32 = (uint32_t)rpr, j32 = (uint32_t)j;        // rows and runs per row are far below 2^31
          const int64_t in_row = (int64_t)((j32 * 61u + j32 / r32) % r32) * 64 + lane;
          i = in_row < words_per_row ? j * words_per_row + in_row : -1;
        } else i = (int64_t)(((unsigned long long)j * (unsigned long long)n_chunks) / (unsigned long long)take) * 64 + lane;
        if (i >= words) i = -1;
      }
      at[u] = i;
      v[u] = i >= 0 ? w[i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < FP_UNROLL; ++u)
      if (at[u] >= 0) h += fp_mix(v[u], (uint32_t)at[u]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o);
  if (lane == 0) red[wv] = h;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long *line = state + (int64_t)z * FP_STATE_WORDS;
    __hip_atomic_store(line + blockIdx.x, red[0] + red[1] + red[2] + red[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence();
    if (atomicAdd(line + FP_BLOCKS + 1, 1ull) == (unsigned long long)(FP_BLOCKS - 1)) {
      __threadfence();
      unsigned long long now = 0;
      for (int i = 0; i < FP_BLOCKS; ++i) now += __hip_atomic_load(line + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      changed[z] = (!store_only && now != line[FP_BLOCKS]) ? 1 : 0;
      line[FP_BLOCKS] = now;
      line[FP_BLOCKS + 1] = 0ull;
    }
  }
}

// out[t][c] = sum of the biases of the decoders that run for target t, sources in ascending order, fp32
template <typename T>
__global__ __launch_bounds__(256) void k_bias_sum(const T *const *b_refs, int64_t d, int64_t L, int tying, uint64_t src_mask,
                                                  float *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= L * d) return;
  const int64_t t = i / d, c = i - t * d;
  float acc = 0.0f;
  if (tying == CLT_TYING_PER_TARGET) {
    acc = Elem<T>::to_f32(b_refs[t][c]);
  } else {
    // six at a time on their way (L = 12: 10.6 -> 7.2 us); a source that is left out stands for the first one that is not
    const uint64_t on = src_mask & ((2ull << t) - 1ull);
    const int64_t some = __ffsll((unsigned long long)on) - 1;
    for (int64_t s0 = 0; on != 0 && s0 <= t; s0 += 6) {
      float b[6];
      uint64_t take = on >> s0;
#pragma unroll
      for (int u = 0; u < 6; ++u) b[u] = Elem<T>::to_f32(b_refs[decoder_slot(tying, (take >> u) & 1ull ? s0 + u : some, t, L)][c]);
#pragma unroll
      for (int u = 0; u < 6; ++u)
        if ((take >> u) & 1ull) acc += b[u];
    }
  }
  out[i] = acc;
}

// [F][pitch] -> [d][F], the way back: decoder z of the slab into the parameter whose address is w_refs[z].
template <typename T>
__global__ __launch_bounds__(256) void k_unpack(const T *src, T *const *w_refs, int64_t d, int64_t F, int64_t pitch) {
  __shared__ T tile[64][65];
  const T *s = src + (int64_t)blockIdx.z * F * pitch;
  T *o = w_refs[blockIdx.z];
  const int64_t f0 = (int64_t)blockIdx.x * 64, d0 = (int64_t)blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    int64_t ff = f0 + i, dd = d0 + tx;
    if (ff < F && dd < d) tile[i][tx] = s[ff * pitch + dd];
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    int64_t dd = d0 + i, ff = f0 + tx;
    if (dd < d && ff < F) o[dd * F + ff] = tile[tx][i];
  }
}

// the same with 4 consecutive elements per access on both sides (d % 4 == 0, F % 4 == 0, 16-byte aligned parameters)
template <typename T>
__global__ __launch_bounds__(256) void k_unpack_vec(const T *__restrict__ src, T *const *__restrict__ w_refs, int64_t d, int64_t F,
                                                    int64_t pitch) {
  __shared__ T tile[64][68];
  const T *s = src + (int64_t)blockIdx.z * F * pitch;
  T *o = w_refs[blockIdx.z];
  const int64_t f0 = (int64_t)blockIdx.x * 64, d0 = (int64_t)blockIdx.y * 64;
  const int q = threadIdx.x & 15, r = threadIdx.x >> 4;
  typedef typename std::conditional<sizeof(T) == 2, uint2, uint4>::type quad_t;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int fl = r + 16 * i;
    const int64_t f = f0 + fl, dd = d0 + q * 4;
    if (f < F && dd < d) *reinterpret_cast<quad_t *>(&tile[fl][q * 4]) = *reinterpret_cast<const quad_t *>(s + f * pitch + dd);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int dl = r + 16 * i;
    const int64_t dd = d0 + dl, f = f0 + q * 4;
    if (dd < d && f < F) {
      T t4[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) t4[k] = tile[q * 4 + k][dl];
      *reinterpret_cast<quad_t *>(o + dd * F + f) = *reinterpret_cast<const quad_t *>(t4);
    }
  }
}

template <typename T, typename OT>
__global__ void k_densify_scatter(const int32_t *row_ptr, const int32_t *col, const T *val, OT *out,
                                  int64_t Tn, int64_t F, int64_t L, int64_t out_layer_stride) {
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int64_t R = L * Tn;
  for (int64_t r = (int64_t)blockIdx.x * nwv + wv; r < R; r += (int64_t)gridDim.x * nwv) {
    const int64_t l = r / Tn, t = r - l * Tn;
    OT *orow = out + l * out_layer_stride + t * F;
    for (int32_t j = row_ptr[r] + lane; j < row_ptr[r + 1]; j += 64) {
      if constexpr (std::is_same<T, OT>::value) orow[col[j]] = val[j];
      else orow[col[j]] = (OT)Elem<T>::to_f32(val[j]);
    }
  }
}

// Dense rows from their lists in one pass: a workgroup puts a piece of a row together in LDS - zeros, then the row's
// survivors - and writes it out 16 bytes per lane.  Bound by the stream of stores.  Element-wise zeros in front of a scatter
// (k_zero_rows, k_densify_scatter; still what rows that are not whole 16-byte pieces take) write at 2 TB/s and touch the
// scattered lines twice.  L = 12, F = 24576, 1000 tokens, bf16 (590 MB): 0.36 -> 0.114 ms.
constexpr int DENSIFY_BYTES = 32 * 1024;   // of LDS: five workgroups per CU

template <typename T, typename OT>
__global__ __launch_bounds__(256) void k_densify_rows(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
                                                      const T *__restrict__ val, OT *__restrict__ out, int64_t Tn, int64_t F, int pieces,
                                                      int64_t out_layer_stride) {
  constexpr int N = DENSIFY_BYTES / (int)sizeof(OT);
  __shared__ __attribute__((aligned(16))) OT piece[N];
  const int64_t r = blockIdx.x / pieces, c0 = (int64_t)(blockIdx.x % pieces) * N;
  const int n = (int)(F - c0 < N ? F - c0 : N), quads = n * (int)sizeof(OT) / 16;
  const int32_t b = row_ptr[r], e = row_ptr[r + 1];
  for (int i = threadIdx.x; i < quads; i += 256) reinterpret_cast<uint4 *>(piece)[i] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  for (int32_t j = b + (int32_t)threadIdx.x; j < e; j += 256) {
    const int64_t c = col[j] - c0;
    if (c < 0 || c >= n) continue;
    if constexpr (std::is_same<T, OT>::value) piece[c] = val[j];
    else piece[c] = (OT)Elem<T>::to_f32(val[j]);
  }
  __syncthreads();
  uint4 *o = reinterpret_cast<uint4 *>(out + r / Tn * out_layer_stride + r % Tn * F + c0);
  for (int i = threadIdx.x; i < quads; i += 256) o[i] = reinterpret_cast<const uint4 *>(piece)[i];
}

// zeros over whole 16-byte pieces
__global__ __launch_bounds__(256) void k_zero_quads(uint4 *out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) out[i] = make_uint4(0u, 0u, 0u, 0u);
}

template <typename OT>
__global__ void k_zero_rows(OT *out, int64_t Tn, int64_t F, int64_t L, int64_t out_layer_stride) {
  const int64_t per_layer = Tn * F;
  const int64_t total = per_layer * L;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    int64_t l = i / per_layer;
    out[l * out_layer_stride + (i - l * per_layer)] = (OT)0;
  }
}

// norms[s][f]: one wavefront per (s, f), summing over the decoders fed by s.
template <typename T>
__global__ __launch_bounds__(256) void k_norms(const T *wp, T *norms, int64_t d, int64_t F, int64_t L, int tying, int64_t pitch) {
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const int64_t total = L * F;
  for (int64_t i = (int64_t)blockIdx.x * nwv + wv; i < total; i += (int64_t)gridDim.x * nwv) {
    const int64_t s = i / F, f = i - s * F;
    float acc = 0.0f;
    const int64_t t0 = s, t1 = tying == CLT_TYING_PER_SOURCE ? s + 1 : L;
    for (int64_t t = t0; t < t1; ++t) {
      const T *row = wp + (decoder_slot(tying, s, t, L) * F + f) * pitch;
      float part = 0.0f;
      for (int64_t o = lane; o < d; o += 64) { float w = Elem<T>::to_f32(row[o]); part = fmaf(w, w, part); }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
      // the reference squares a norm that was rounded to the model dtype (decoder.py:452)
      float nrm = Elem<T>::round(sqrtf(part));
      acc += Elem<T>::round(nrm * nrm);
    }
    if (lane == 0) norms[i] = Elem<T>::from_f32(sqrtf(acc));
  }
}

// acc[tok][f] = round(acc[tok][f] + v') over the survivors (f, v) of one layer: the running sum of
// activations that decoders tied per target consume (reference clt/models/decoder.py:208-246), every
// addition rounded to the model dtype as the reference's `summed_activation += activation_tensor` is.
// One wavefront per token row; a row's columns are distinct, so no two lanes touch one element.
template <typename T>
__global__ __launch_bounds__(256) void k_accumulate_dense(const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
                                                          const T *__restrict__ val, const T *__restrict__ foff,
                                                          const T *__restrict__ fscale, T *__restrict__ acc, int64_t Tn,
                                                          int64_t F, int64_t layer, int init) {
  const int lane = lane_id(), wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  for (int64_t tok = (int64_t)blockIdx.x * nwv + wv; tok < Tn; tok += (int64_t)gridDim.x * nwv) {
    const int64_t r = layer * Tn + tok;
    T *arow = acc + tok * F;
    for (int32_t j = row_ptr[r] + lane; j < row_ptr[r + 1]; j += 64) {
      const int32_t f = col[j];
      float v = Elem<T>::to_f32(val[j]);
      if (v != 0.0f) {   // the affine terms apply to the selected (non-zero) entries only
        if (foff) v = Elem<T>::round(v + Elem<T>::to_f32(foff[f]));
        if (fscale) v = Elem<T>::round(v * Elem<T>::to_f32(fscale[f]));
      }
      const float old = init ? 0.0f : Elem<T>::to_f32(arow[f]);
      arow[f] = Elem<T>::from_f32(old + v);
    }
  }
}

constexpr int DEC_SLICES = 8;  // one feature slice per XCD of an MI355X

// Partial rows of a batch, in units of Tn rows of d: a target's feature slices, or for a short batch (whose rows then stay
// below PAIR_BYTES) the pairs' of a launch over all sources with two slices.
constexpr int64_t PAIR_BYTES = 256 << 20;
static int64_t partial_rows(int64_t Tn, int64_t d, int64_t L) {
  const int64_t by_target = DEC_SLICES * L, by_pair = L * (L + 1);
  return by_pair > by_target && by_pair * Tn * d * 4 <= PAIR_BYTES ? by_pair : by_target;
}
static bool one_launch(int64_t Tn, int64_t d, int64_t L, int slices) {
  const int64_t rows = slices * (L * (L + 1) / 2);
  return rows <= partial_rows(Tn, d, L) && rows * Tn * d * 4 <= PAIR_BYTES;
}

static size_t partial_bytes(int64_t Tn, int64_t d, int64_t L) {
  return ((size_t)partial_rows(Tn, d, L) * Tn * d * 4 + 255) & ~(size_t)255;
}

static size_t decode_ws_bytes(int64_t Tn, int64_t d, int64_t L) {
  size_t part = partial_bytes(Tn, d, L);
  size_t sp = ((size_t)L * Tn * (DEC_SLICES + 1) * 4 + 255) & ~(size_t)255;
  return part + sp;
}

// feature slices of the line schedule: F x 128 bytes per slice must stay inside an L2
static int line_slices(int64_t F) { return (int)clt_ceil_div(F * 128, LINE_L2_BYTES); }
// The quarter schedule keeps F / QUARTER_SLICES rows x a quarter of the columns per XCD: it is taken while
// that stays near one 4 MiB L2 (measured: 4.7 MiB at F = 24576, d = 768 bf16 is still 2 % ahead of the line
// schedule, 8.4 MiB at F = 32768, d = 1024 is 25 % behind it)
constexpr int64_t QUARTER_L2_BYTES = 5 << 20;
static bool quarter_fits(int64_t F, int64_t d, int elem_bytes) {
  return (F / QUARTER_SLICES) * (d / QUARTER_PARTS) * elem_bytes <= QUARTER_L2_BYTES;
}

static bool quarter_shape_ok(int64_t d, int elem_bytes) {
  const int V = 16 / elem_bytes;
  const int per_lane = (int)(d / 64), hq = per_lane / V;
  const bool htail = (per_lane % V) != 0;
  if (elem_bytes == 2) return (hq == 1) || (hq == 2 && !htail) || (hq == 4 && !htail);
  return (hq == 2 || hq == 3 || hq == 4) && !htail;
}

// Which schedule launch_decode takes; `ws_ok`: a workspace of decode_ws_bytes(), 256-byte aligned;
// `wp_ok`: the packed decoders are 16-byte aligned.
static int plan_route(int64_t d, int64_t F, int tying, int elem_bytes, bool ws_ok, bool wp_ok) {
  const int V = 16 / elem_bytes;
  const int64_t chunk = 64 * V, nf = d / chunk, rem = d % chunk;
  const bool can_slice = ws_ok && (d % 4 == 0) && F >= 64 * DEC_SLICES;
  const bool fast = (d % V == 0) && wp_ok && nf <= 4 && (nf > 0 || rem > 0);
  if (fast && can_slice && tying != CLT_TYING_PER_TARGET && d % 256 == 0 && F >= 64 * QUARTER_SLICES &&
      quarter_shape_ok(d, elem_bytes) && quarter_fits(F, d, elem_bytes))
    return CLT_ROUTE_QUARTER;
  // the line schedule takes any width that is a whole number of cache lines
  if (can_slice && wp_ok && tying != CLT_TYING_PER_TARGET && (d * elem_bytes) % 128 == 0 && line_slices(F) <= DEC_SLICES)
    return CLT_ROUTE_LINE;
  if (!fast) return CLT_ROUTE_GENERIC;
  if (!can_slice) return CLT_ROUTE_SINGLE;
  return tying == CLT_TYING_PER_TARGET ? CLT_ROUTE_SLICED_ALL_SOURCES : CLT_ROUTE_SLICED;
}

template <typename T>
static int launch_decode(const int32_t *row_ptr, const int32_t *col, const void *val, const void *wp,
                         const float *bias_sum, const void *foff, const void *fscale, const float *skip_add,
                         void *out, int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin,
                         int64_t t_end, uint64_t src_mask, int out_f32, void *workspace, size_t workspace_bytes,
                         hipStream_t stream) {
  constexpr int V = WVec<T>::V;
  const int nwv = 4;
  const int64_t pitch = clt_pitch(d, (int)sizeof(T));
  const int64_t blocks_per_t = clt_ceil_div(Tn, nwv);
  const bool can_slice = workspace && workspace_bytes >= decode_ws_bytes(Tn, d, L) && (d % 4 == 0) &&
                         F >= 64 * DEC_SLICES && ((((uintptr_t)workspace) & 255u) == 0);
  const int ns = can_slice ? DEC_SLICES : 1;
  int32_t *sptr = nullptr; float *partial = nullptr;
  if (can_slice) {
    partial = (float *)workspace;
    sptr = (int32_t *)((char *)workspace + partial_bytes(Tn, d, L));
  }
  int64_t nblk = blocks_per_t * (t_end - t_begin);
  if (nblk <= 0) return CLT_OK;
  if (nblk > 2147483647LL) return CLT_ERR_RANGE;
  const bool affine = foff || fscale;
  const bool few = Tn * (t_end - t_begin) <= DECODE_FEW;
  const int64_t chunk = 64 * V;
  const int64_t nf = d / chunk, rem = d % chunk;
  const bool fast = (d % V == 0) && clt_aligned16(wp) && nf <= 4 && (nf > 0 || rem > 0);
  const int route = plan_route(d, F, tying, (int)sizeof(T), can_slice, clt_aligned16(wp));
  if (can_slice && !fast && route != CLT_ROUTE_LINE)
    return launch_decode<T>(row_ptr, col, val, wp, bias_sum, foff, fscale, skip_add, out, Tn, d, F,
                            L, tying, t_begin, t_end, src_mask, out_f32, nullptr, 0, stream);
#define CLT_DEC_ARGS(FO, FS)                                                                                    \
  row_ptr, col, (const T *)val, (const T *)wp, bias_sum, FO, FS, skip_add, out, Tn, d, F, L, tying, tb,         \
      t_end, src_mask, out_f32, sptr, partial, ns, src, pitch
#define CLT_DEC(NFN, TL, UN)                                                                                    \
  do {                                                                                                          \
    if (affine && can_slice)                                                                                    \
      k_decode<T, NFN, TL, UN, true, true><<<(unsigned)nblk, 256, 0, stream>>>(CLT_DEC_ARGS((const T *)foff, (const T *)fscale)); \
    else if (affine)                                                                                            \
      k_decode<T, NFN, TL, UN, true, false><<<(unsigned)nblk, 256, 0, stream>>>(CLT_DEC_ARGS((const T *)foff, (const T *)fscale)); \
    else if (can_slice)                                                                                         \
      k_decode<T, NFN, TL, UN, false, true><<<(unsigned)nblk, 256, 0, stream>>>(CLT_DEC_ARGS(nullptr, nullptr)); \
    else if (few && NFN < 4)                                                                                    \
      k_decode<T, NFN, TL, decode_few_in_flight<T, NFN, TL>(), false, false><<<(unsigned)(Tn * (t_end - t_begin)), 64, 0, stream>>>(CLT_DEC_ARGS(nullptr, nullptr)); \
    else                                                                                                        \
      k_decode<T, NFN, TL, UN, false, false><<<(unsigned)nblk, 256, 0, stream>>>(CLT_DEC_ARGS(nullptr, nullptr)); \
  } while (0)
#define CLT_DEC_TAIL(NFN, UN)                              \
  do {                                                     \
    if (rem == 0) CLT_DEC(NFN, 0, UN);                     \
    else if (rem * 2 == chunk) CLT_DEC(NFN, 1, UN);        \
    else CLT_DEC(NFN, 2, UN);                              \
  } while (0)
  // (source, target) pairs of a launch over all sources
  int64_t n_pairs = 0;
  for (int64_t s = 0; s < t_end; ++s)
    if ((src_mask >> s) & 1ull) n_pairs += t_end - (s > t_begin ? s : t_begin);
  // quarter-row schedule: 2 feature slices x 4 column quarters (see k_decode_quarter)
  bool quartered = false; int quarter_ns = QUARTER_SLICES;
  const bool quarter_pairs = one_launch(Tn, d, L, QUARTER_SLICES);
  if (route == CLT_ROUTE_LINE) {
    constexpr int ntok = 2;                               // tokens per wavefront
    const UnitPlan lp = make_unit_plan(line_slices(F), (int)(d * (int64_t)sizeof(T) / 128), Tn, nwv * ntok);
    // one 32-bit word per survivor and 32-bit row offsets: feature index below 2^16, matrix below 4 GiB
    const bool pack = sizeof(T) == 2 && F <= 65536 && F * pitch * (int64_t)sizeof(T) < (1ll << 32);
    k_slice_ptr<<<1024, 256, 0, stream>>>(row_ptr, col, L * Tn, F, lp.ns, sptr);
    const bool pairs = one_launch(Tn, d, L, lp.ns);
    for (int src = pairs ? -1 : 0; src < (pairs ? 0 : (int)t_end); ++src) {
      if (!pairs && !((src_mask >> src) & 1ull)) continue;
      const int64_t tb = src > t_begin ? src : t_begin;
      const int64_t lb = 8 * (int64_t)lp.bpx * (pairs ? n_pairs : t_end - tb);
      if (lb <= 0) continue;
      if (lb > 2147483647LL) return CLT_ERR_RANGE;
#define CLT_DECL(AF, PK, NT)                                                                                          \
  k_decode_line<T, AF, PK, NT><<<(unsigned)lb, 256, 0, stream>>>(col, (const T *)val, (const T *)wp, (const T *)foff, \
      (const T *)fscale, Tn, d, F, L, tying, tb, src_mask, sptr, partial, src, lp, pitch, t_end)
#define CLT_DECL2(AF, PK) CLT_DECL(AF, PK, ntok)
      if (affine) { if (pack) CLT_DECL2(true, true); else CLT_DECL2(true, false); }
      else { if (pack) CLT_DECL2(false, true); else CLT_DECL2(false, false); }
#undef CLT_DECL2
#undef CLT_DECL
    }
    k_decode_reduce<T><<<2048, 256, 0, stream>>>(partial, bias_sum, skip_add, out, Tn, d, L, t_begin, t_end, lp.ns, out_f32, src_mask, pairs);
    return clt_check_launch();
  }
  if (route == CLT_ROUTE_QUARTER) {
    const int per_lane = (int)(d / 64);                    // columns per lane
    const int hq = per_lane / V, htail = (per_lane % V) != 0;
    // feature slices: F / qs rows x a quarter of the columns per XCD at a time, about one L2
    const int qs = QUARTER_SLICES;
    const UnitPlan up = make_unit_plan(qs, QUARTER_PARTS, Tn, nwv * QUARTER_NTOK);
    // one 32-bit word per survivor and 32-bit row offsets: feature index below 2^16, matrix below 4 GiB
    const bool qpack = sizeof(T) == 2 && F <= 65536 && F * pitch * (int64_t)sizeof(T) < (1ll << 32);
#define CLT_DECQ(HQN, HTN, UN)                                                                                       \
  do {                                                                                                               \
    k_slice_ptr<<<1024, 256, 0, stream>>>(row_ptr, col, L * Tn, F, qs, sptr);                                        \
    for (int src = quarter_pairs ? -1 : 0; src < (quarter_pairs ? 0 : (int)t_end); ++src) {                          \
      if (!quarter_pairs && !((src_mask >> src) & 1ull)) continue;                                                   \
      const int64_t tb = src > t_begin ? src : t_begin;                                                              \
      const int64_t qb = 8 * (int64_t)up.bpx * (quarter_pairs ? n_pairs : t_end - tb);                               \
      if (qb <= 0) continue;                                                                                         \
      if (qb > 2147483647LL) return CLT_ERR_RANGE;                                                                   \
      if (affine) k_decode_quarter<T, HQN, HTN, UN, true, false><<<(unsigned)qb, 256, 0, stream>>>(col, (const T *)val, (const T *)wp, \
          (const T *)foff, (const T *)fscale, Tn, d, F, L, tying, tb, src_mask, sptr, partial, src, pitch, up, t_end);      \
      else if (qpack) k_decode_quarter<T, HQN, HTN, UN, false, sizeof(T) == 2><<<(unsigned)qb, 256, 0, stream>>>(col, (const T *)val, (const T *)wp, \
          nullptr, nullptr, Tn, d, F, L, tying, tb, src_mask, sptr, partial, src, pitch, up, t_end);                        \
      else k_decode_quarter<T, HQN, HTN, UN, false, false><<<(unsigned)qb, 256, 0, stream>>>(col, (const T *)val, (const T *)wp, \
          nullptr, nullptr, Tn, d, F, L, tying, tb, src_mask, sptr, partial, src, pitch, up, t_end);                        \
    }                                                                                                                \
    quartered = true; quarter_ns = qs;                                                                               \
  } while (0)
    if constexpr (sizeof(T) == 2) {
      if (hq == 1 && !htail) CLT_DECQ(1, 0, 2);
      else if (hq == 1 && htail) CLT_DECQ(1, 1, 2);
      else if (hq == 2 && !htail) CLT_DECQ(2, 0, 2);
      else if (hq == 4 && !htail) CLT_DECQ(4, 0, 2);
    } else {
      if (hq == 2 && !htail) CLT_DECQ(2, 0, 2);
      else if (hq == 3 && !htail) CLT_DECQ(3, 0, 2);
      else if (hq == 4 && !htail) CLT_DECQ(4, 0, 2);
    }
#undef CLT_DECQ
  }
  if (quartered) {
    k_decode_reduce<T><<<2048, 256, 0, stream>>>(partial, bias_sum, skip_add, out, Tn, d, L, t_begin, t_end, quarter_ns, out_f32, src_mask, quarter_pairs);
    return clt_check_launch();
  }
  if (can_slice) k_slice_ptr<<<1024, 256, 0, stream>>>(row_ptr, col, L * Tn, F, ns, sptr);
  if (fast) {
    // sliced: one launch per source layer, targets max(src, t_begin) .. t_end-1
    // decoders tied per target: one launch, sources walked inside the wavefront (src = -1)
    const bool all_src = can_slice && tying == CLT_TYING_PER_TARGET;
    const int n_launch = all_src ? 1 : (can_slice ? (int)t_end : 1);
    for (int src0 = 0; src0 < n_launch; ++src0) {
      const int src = all_src ? -1 : src0;
      int64_t tb = t_begin;
      if (all_src) {
        nblk = clt_ceil_div(Tn, nwv * SLICED_NTOK) * (t_end - tb) * ns;
        if (nblk > 2147483647LL) return CLT_ERR_RANGE;
      } else if (can_slice) {
        if (!((src_mask >> src) & 1ull)) continue;
        if (src > tb) tb = src;
        nblk = clt_ceil_div(Tn, nwv * SLICED_NTOK) * (t_end - tb) * ns;
        if (nblk <= 0) continue;
        if (nblk > 2147483647LL) return CLT_ERR_RANGE;
      }
      if (nf == 0) CLT_DEC(0, 2, 8);
      else if (nf == 1) CLT_DEC_TAIL(1, 8);
      else if (nf == 2) CLT_DEC_TAIL(2, 6);
      else if (nf == 3) CLT_DEC_TAIL(3, 4);
      else if (rem == 0) CLT_DEC(4, 0, 4);
      else CLT_DEC(4, 2, 2);
    }
  } else {
    const int64_t tb = t_begin; const int src = 0; (void)tb; (void)src;
    k_decode_generic<T><<<(unsigned)nblk, 256, 0, stream>>>(row_ptr, col, (const T *)val, (const T *)wp, bias_sum,
        (const T *)foff, (const T *)fscale, skip_add, out, Tn, d, F, L, tying, t_begin, t_end, src_mask, out_f32, pitch);
  }
#undef CLT_DEC_TAIL
#undef CLT_DEC
#undef CLT_DEC_ARGS
  if (can_slice)
    k_decode_reduce<T><<<2048, 256, 0, stream>>>(partial, bias_sum, skip_add, out, Tn, d, L, t_begin, t_end, ns, out_f32, src_mask);
  return clt_check_launch();
}

}  // namespace

template <typename T>
static int launch_decode_thin(const int32_t *row_ptr, const int32_t *col, const void *val, const void *wp, const float *bias_sum,
                              const float *skip_add, void *out, int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin,
                              int64_t t_end, uint64_t src_mask, int out_f32, int64_t max_entries, hipStream_t stream) {
  constexpr int V = WVec<T>::V;
  const int64_t blocks = 8 * clt_ceil_div((Tn + 1) / 2, THIN_WAVES) * (t_end - t_begin);
  if (blocks > 2147483647LL) return CLT_ERR_RANGE;
  const int hq = (int)(d / 64) / V, htail = ((int)(d / 64) % V) != 0;
#define CLT_THIN(HQN, HTN)                                                                                            \
  k_decode_thin<T, HQN, HTN><<<(unsigned)blocks, THIN_WAVES * 64, 0, stream>>>(row_ptr, col, (const T *)val, (const T *)wp, bias_sum, \
      skip_add, out, Tn, d, F, L, tying, t_begin, t_end, src_mask, out_f32, clt_pitch(d, (int)sizeof(T)), max_entries)
  if constexpr (sizeof(T) == 2) {
    if (hq == 1 && !htail) CLT_THIN(1, 0);
    else if (hq == 1) CLT_THIN(1, 1);
    else if (hq == 2) CLT_THIN(2, 0);
    else CLT_THIN(4, 0);
  } else {
    if (hq == 2) CLT_THIN(2, 0);
    else if (hq == 3) CLT_THIN(3, 0);
    else CLT_THIN(4, 0);
  }
#undef CLT_THIN
  const int units = (int)(d / (8 * V));
  k_decode_thin_longest<T><<<(unsigned)(THIN_PARTS * units * (t_end - t_begin)), THIN_WAVES * 64, 0, stream>>>(row_ptr, col, (const T *)val,
      (const T *)wp, bias_sum, skip_add, out, Tn, d, F, L, tying, t_end, src_mask, out_f32, clt_pitch(d, (int)sizeof(T)), units, max_entries);
  return clt_check_launch();
}

// What k_decode_thin takes: row numbers over all decoders in 32 bits, rows in quarters that a lane group reads whole.
static bool decode_thin_ok(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int tying, int dtype) {
  if (!clt_model_dtype(dtype) || (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE)) return false;
  if (T <= 0 || F <= 0 || L <= 0 || L > 64 || targets <= 0 || targets > L || d <= 0 || d % 256 != 0) return false;
  const int64_t n_dec = tying == CLT_TYING_NONE ? L * (L + 1) / 2 : L;
  return quarter_shape_ok(d, clt_elem_bytes(dtype)) && n_dec * F <= 0x7FFFFFFFll && L * T < 0x7FFFFFFFll;
}

// What the gathers move: bytes of decoder rows, bytes of those that some token refers to, (source, target, token) triples.
struct GatherWork { double bytes, distinct, triples; };
static GatherWork gather_work(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying, int dtype) {
  const double row = (double)d * clt_elem_bytes(dtype), pairs = 0.5 * targets * (2 * L - targets + 1), list = (double)entries / L;
  GatherWork g;
  g.bytes = list * pairs * row;
  g.distinct = (tying == CLT_TYING_NONE ? pairs : (double)L) * F * (1.0 - exp(-list / F)) * row;
  g.triples = pairs * T;
  return g;
}

// What the prices of the decodes were measured at: 6006 shapes at random (L 2 - 16, d 256 - 2048, F 1024 - 32768, T 32 - 8192, 1 - 256
// survivors per source and token, untied and tied per source), lists of equal length, lists with the heavy tokens of a top-k over the batch
// and thresholds.  At 3753 other shapes the choice costs, against the best of the three, 1.2 % (float32) and 1.9 % (16 bits) for threshold
// lists, 6.0 and 7.7 % for a top-k's; while each decode was priced from shapes of its own it cost 3.8, 3.3, 8.3 and 8.6 %.
//
// The schedules by sources: bytes per us of decoder rows out of the L2s, of fp32 partial rows written and read, of rows from HBM that some
// token refers to, and us per source for its launches; off by 8 - 11 % in the mean.  With too little work for those (the lines of
// engine._wants_sliced_decode) a wavefront walks a row's whole list: lists of equal length then take two thirds of the mean, heavy tokens
// more, and the price is put a tenth below it.  In 16 bits, where a threshold list's total is the last batch's, the price by sources bounds
// it there, so that small batches do not change route, and with it their rounding, from one call to the next.
double clt_decode_gather_us(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying, int dtype) {
  const int esz = clt_elem_bytes(dtype);
  const bool wide = dtype == CLT_F32;
  const GatherWork g = gather_work(T, d, F, L, targets, entries, tying, dtype);
  const int64_t n_dec = tying == CLT_TYING_NONE ? L * (L + 1) / 2 : L;
  const double partial = g.triples * (double)d * 16;
  if (T * targets < 8192 && n_dec * F * clt_pitch(d, esz) * esz < (128ll << 20) && d * esz < 5 * 1024) {
    const double list = (double)entries / T;
    if (wide) return 7.7 + g.bytes / 10.3e6 + g.distinct / 3.8e6 + list * 0.086;
    const double walk = 11.2 + g.bytes / 11.5e6 + g.distinct / 5e6 + list * 0.111, sources = 0.3 * L + g.bytes / 18.1e6 + partial / 4.5e6 + g.distinct / 5.5e6;
    return walk < sources ? walk : sources;
  }
  if (wide) {
    const bool quarter = plan_route(d, F, tying, esz, true, true) == CLT_ROUTE_QUARTER;
    return 11.5 + 0.4 * L + g.bytes / 23.5e6 + partial / (quarter ? 4e6 : 2.4e6) + g.distinct / 7.9e6;
  }
  return 14.5 + 0.3 * L + g.bytes / 20.4e6 + partial / 4e6 + g.distinct / 8.1e6;
}

// Against the schedules by sources (k_decode_quarter, k_decode_line), which move rows at 17 TB/s out of the L2s, bring each one there
// from HBM and read and write the partial rows of every triple, and against the decodes from LDS tiles.  This kernel, from what it
// measured (bf16 and float32; L 2 - 16, d 512 - 2048, F 1024 - 24576, T 32 - 8000, 1 - 200 survivors per source and token): 9.5
// TB/s, as much time again for a row's first use, 0.25 ns per triple, and no less than a workgroup's chain over its lists, or over
// one of 4000 entries, as a top-k over the batch may give a single token (k_decode_thin_longest says what longer ones cost).  Within 15 %, but for rows used more than
// 20 times, which it does faster; against the tiles a third more is let pass, because lists of equal length take that much less here than the mean (bf16,
// T = 153, L = 12, d = 2048, F = 5224, 35 per token: 244 / 354 of the tiles; float32, 522, 9, 1024, 2960, 18: 167 / 278).  us, schedule by sources / this: T = 3000, L = 12, F = 24576, d = 768, bf16, 200 survivors per
// token over all layers 1530 / 854, 20 695 / 224; per layer 16: 1253 / 747; T = 1000, 50: 1100 / 790; T = 300, 200: 877 / 1078;
// T = 77, 200: 340 / 356; float32, T = 600, 200: 2790 / 3910.
extern "C" int clt_decode_thin_wanted(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying, int dtype) {
  if (entries < 0 || !decode_thin_ok(T, d, F, L, targets, tying, dtype)) return 0;
  const GatherWork g = gather_work(T, d, F, L, targets, entries, tying, dtype);
  const double flow = g.bytes / 9.5e6 + g.distinct / 10e6 + g.triples * 0.25e-3, longest = entries < 4000 ? (double)entries : 4000.0;
  const double chain = 0.1 * (double)entries / T > 0.025 * longest ? 0.1 * (double)entries / T : 0.025 * longest;
  const double thin = (flow > chain ? flow : chain) + 18;
  return thin < 0.95 * (g.bytes / 17e6 + g.distinct / 6.3e6 + g.triples * (double)d * 16 / 3.2e6 + 5) &&
         thin < 1.3 * clt_decode_tiles_us(T, d, F, L, targets, entries, tying, dtype) &&
         thin < 1.3 * clt_decode_rows_us(T, d, F, L, targets, entries, tying, dtype);
}

// max_entries < 0: whatever the lists hold
static int decode_thin(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed, const float *bias_sum,
                       const float *skip_add, void *out, int64_t T, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin,
                       int64_t t_end, uint64_t src_mask, int dtype, int out_f32, int64_t max_entries, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T < 0 || t_begin < 0 || t_end > L || t_begin > t_end) return CLT_ERR_ARG;
  if (T == 0 || t_begin == t_end) return CLT_OK;
  if (!decode_thin_ok(T, d, F, L, t_end - t_begin, tying, dtype)) return CLT_ERR_ARG;
  if (!row_ptr || !col || !val || !w_packed || !out) return CLT_ERR_ARG;
  if (!clt_aligned16(w_packed) || !clt_aligned16(out) || (bias_sum && !clt_aligned16(bias_sum)) || (skip_add && !clt_aligned16(skip_add)))
    return CLT_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == CLT_BF16)
    return launch_decode_thin<bf16_t>(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, max_entries, s);
  if (dtype == CLT_F16)
    return launch_decode_thin<f16_t>(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, max_entries, s);
  return launch_decode_thin<float>(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, max_entries, s);
}

extern "C" int clt_decode_thin(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed,
                               const float *bias_sum, const float *skip_add, void *out, int64_t T, int64_t d, int64_t F,
                               int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int dtype, int out_f32,
                               void *stream) {
  return decode_thin(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, dtype, out_f32, -1, stream);
}

extern "C" int clt_decode_thin_up_to(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed,
                                     const float *bias_sum, const float *skip_add, void *out, int64_t T, int64_t d, int64_t F,
                                     int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int dtype, int out_f32,
                                     int64_t max_entries, void *stream) {
  if (max_entries < 0) return CLT_ERR_ARG;
  return decode_thin(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, dtype, out_f32, max_entries, stream);
}

extern "C" size_t clt_decode_workspace_bytes(int64_t T, int64_t d, int64_t F, int64_t L) {
  (void)F;
  if (T <= 0 || d <= 0 || L <= 0) return 256;
  return decode_ws_bytes(T, d, L);
}

extern "C" int clt_decode_sparse(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed,
                                 const float *bias_sum, const void *feat_offset, const void *feat_scale,
                                 const float *skip_add, void *out, int64_t T, int64_t d, int64_t F, int64_t L,
                                 int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int dtype,
                                 int out_f32, void *workspace, size_t workspace_bytes, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T < 0 || d <= 0 || F <= 0 || L <= 0 || L > 64) return CLT_ERR_ARG;
  if (t_begin < 0 || t_end > L || t_begin > t_end) return CLT_ERR_ARG;
  if (tying < 0 || tying > 2) return CLT_ERR_ARG;
  if (T == 0 || t_begin == t_end) return CLT_OK;
  if (!row_ptr || !w_packed || !out) return CLT_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == CLT_BF16)
    return launch_decode<bf16_t>(row_ptr, col, val, w_packed, bias_sum, feat_offset, feat_scale, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, workspace, workspace_bytes, s);
  if (dtype == CLT_F16)
    return launch_decode<f16_t>(row_ptr, col, val, w_packed, bias_sum, feat_offset, feat_scale, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, workspace, workspace_bytes, s);
  return launch_decode<float>(row_ptr, col, val, w_packed, bias_sum, feat_offset, feat_scale, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, workspace, workspace_bytes, s);
}

template <typename T>
static int launch_decode_over(const int32_t *row_ptr, const int32_t *col, const void *val, const void *wp, const float *bias_sum,
                              const float *skip_add, void *out, int64_t Tn, int64_t d, int64_t F, int64_t L, int tying, int64_t t_begin,
                              int64_t t_end, uint64_t src_mask, int out_f32, int64_t only_above, hipStream_t stream) {
  const int64_t pitch = clt_pitch(d, 2);
  const int units = (int)(d / 64);
  // tokens of a workgroup: the workgroups of an XCD share the tokens of one unit
  const int64_t share = clt_ceil_div(Tn, OVER_BLOCKS / 8 * OVER_WAVES) * OVER_WAVES;
  const int ntok = share < OVER_TOKENS ? (int)share : OVER_TOKENS;
  const UnitPlan lp = make_unit_plan(1, units, Tn, ntok);
  const int64_t blocks = 8 * (int64_t)lp.bpx * (t_end - t_begin);
  const unsigned grid = (unsigned)(blocks < OVER_BLOCKS ? blocks : OVER_BLOCKS);
  const int lds = ntok * 64 * (int)sizeof(float);
  // one 32-bit word per survivor and 32-bit row offsets: feature index below 2^16, matrix below 4 GiB
  const bool pack = F <= 65536 && F * pitch * 2 < (1ll << 32);
  const void *k = pack ? (const void *)k_decode_over<T, true> : (const void *)k_decode_over<T, false>;
  if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return CLT_ERR_LAUNCH;
#define CLT_OVER(PK)                                                                                                             \
  k_decode_over<T, PK><<<grid, OVER_WAVES * 64, lds, stream>>>(row_ptr, col, (const T *)val, (const T *)wp, bias_sum, skip_add,  \
                                                               out, Tn, d, F, L, tying, (int)t_end, src_mask, out_f32, lp, ntok, \
                                                               pitch, blocks, only_above)
  if (pack) CLT_OVER(true); else CLT_OVER(false);
#undef CLT_OVER
  return clt_check_launch();
}

extern "C" int clt_decode_sparse_if_over(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed,
                                         const float *bias_sum, const float *skip_add, void *out, int64_t T, int64_t d,
                                         int64_t F, int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask,
                                         int dtype, int out_f32, int64_t max_entries, void *stream) {
  if (dtype != CLT_BF16 && dtype != CLT_F16) return CLT_ERR_DTYPE;
  if (T < 0 || d <= 0 || F <= 0 || L <= 0 || L > 64 || d % 64 != 0 || max_entries < 0) return CLT_ERR_ARG;
  if (t_begin < 0 || t_end > L || t_begin > t_end) return CLT_ERR_ARG;
  if (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE) return CLT_ERR_ARG;
  if (T == 0 || t_begin == t_end) return CLT_OK;
  if (!row_ptr || !w_packed || !out) return CLT_ERR_ARG;
  if (!clt_aligned16(w_packed)) return CLT_ERR_ALIGN;
  if (T * (d / 64) > 0x7FFFFFFFll) return CLT_ERR_RANGE;       // blocks of a target
  const auto run = dtype == CLT_BF16 ? launch_decode_over<bf16_t> : launch_decode_over<f16_t>;
  return run(row_ptr, col, val, w_packed, bias_sum, skip_add, out, T, d, F, L, tying, t_begin, t_end, src_mask, out_f32, max_entries,
             (hipStream_t)stream);
}

extern "C" int clt_pack_decoder(const void *w_ref, void *w_packed, int64_t d, int64_t F, int64_t n_dec,
                                int64_t in_stride, int64_t out_stride, int dtype, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || F <= 0 || n_dec < 0 || n_dec > 65535) return CLT_ERR_ARG;
  if (n_dec == 0) return CLT_OK;
  if (!w_ref || !w_packed) return CLT_ERR_ARG;
  dim3 grid((unsigned)clt_ceil_div(F, 64), (unsigned)clt_ceil_div(d, 64), (unsigned)n_dec);
  if (clt_ceil_div(d, 64) > 65535) return CLT_ERR_RANGE;
  hipStream_t s = (hipStream_t)stream;
  if (dtype != CLT_F32) k_pack<bf16_t><<<grid, 256, 0, s>>>((const bf16_t *)w_ref, (bf16_t *)w_packed, d, F, in_stride, out_stride, clt_pitch(d, 2));
  else k_pack<float><<<grid, 256, 0, s>>>((const float *)w_ref, (float *)w_packed, d, F, in_stride, out_stride, clt_pitch(d, 4));
  return clt_check_launch();
}

extern "C" int clt_decoder_fingerprint(void *const *w_refs_dev, int64_t n_dec, int64_t d, int64_t F, int dtype,
                                       uint64_t *state, int32_t *changed, int store_only, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || F <= 0 || n_dec < 0 || n_dec > 65535) return CLT_ERR_ARG;
  if (n_dec == 0) return CLT_OK;
  if (!w_refs_dev || !state || !changed) return CLT_ERR_ARG;
  const int64_t words = d * F * clt_elem_bytes(dtype) / 4;     // a last odd 16-bit element is not looked at
  if (words <= 0) return CLT_ERR_ARG;
  const int64_t row_bytes = F * clt_elem_bytes(dtype);
  if ((((uintptr_t)state) & 127u) != 0) return CLT_ERR_ALIGN;
  k_fingerprint<<<dim3(FP_BLOCKS, (unsigned)n_dec), 256, 0, (hipStream_t)stream>>>(
      (const uint32_t *const *)w_refs_dev, words, d, row_bytes % 4 == 0 ? row_bytes / 4 : 0,
      (unsigned long long *)state, changed, store_only);
  return clt_check_launch();
}

extern "C" int clt_pack_decoders_if(void *const *w_refs_dev, void *w_packed, int64_t n_dec, int64_t d, int64_t F,
                                    int dtype, const int32_t *changed, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || F <= 0 || n_dec < 0 || n_dec > 65535) return CLT_ERR_ARG;
  if (n_dec == 0) return CLT_OK;
  if (!w_refs_dev || !w_packed || !changed) return CLT_ERR_ARG;
  const dim3 grid(FP_PACK_BLOCKS, (unsigned)n_dec);
  hipStream_t s = (hipStream_t)stream;
  if (dtype != CLT_F32) k_pack_if<bf16_t><<<grid, 256, 0, s>>>((bf16_t *const *)w_refs_dev, (bf16_t *)w_packed, d, F, clt_pitch(d, 2), changed);
  else k_pack_if<float><<<grid, 256, 0, s>>>((float *const *)w_refs_dev, (float *)w_packed, d, F, clt_pitch(d, 4), changed);
  return clt_check_launch();
}

extern "C" int clt_bias_sum(void *const *b_refs_dev, int64_t n_dec, int64_t d, int64_t L, int tying, uint64_t src_mask,
                            int dtype, float *out, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || L <= 0 || L > 64 || tying < 0 || tying > 2 || !b_refs_dev || !out) return CLT_ERR_ARG;
  if (n_dec != (tying == CLT_TYING_NONE ? L * (L + 1) / 2 : L)) return CLT_ERR_ARG;
  const unsigned nb = (unsigned)clt_ceil_div(L * d, 256);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == CLT_BF16) k_bias_sum<bf16_t><<<nb, 256, 0, s>>>((const bf16_t *const *)b_refs_dev, d, L, tying, src_mask, out);
  else if (dtype == CLT_F16) k_bias_sum<f16_t><<<nb, 256, 0, s>>>((const f16_t *const *)b_refs_dev, d, L, tying, src_mask, out);
  else k_bias_sum<float><<<nb, 256, 0, s>>>((const float *const *)b_refs_dev, d, L, tying, src_mask, out);
  return clt_check_launch();
}

extern "C" int clt_unpack_decoders(const void *w_packed, void *const *w_refs_dev, void *const *w_refs_host, int64_t n_dec,
                                   int64_t d, int64_t F, int dtype, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || F <= 0 || n_dec < 0 || n_dec > 65535) return CLT_ERR_ARG;
  if (n_dec == 0) return CLT_OK;
  if (!w_packed || !w_refs_dev) return CLT_ERR_ARG;
  if (clt_ceil_div(d, 64) > 65535) return CLT_ERR_RANGE;
  dim3 grid((unsigned)clt_ceil_div(F, 64), (unsigned)clt_ceil_div(d, 64), (unsigned)n_dec);
  hipStream_t s = (hipStream_t)stream;
  // w_refs_host (optional): the same addresses on the host, to see whether the 4-element kernel may be used
  bool vec = w_refs_host != nullptr && d % 4 == 0 && F % 4 == 0;
  for (int64_t i = 0; vec && i < n_dec; ++i) vec = clt_aligned16(w_refs_host[i]);
  if (vec) {
    if (dtype != CLT_F32) k_unpack_vec<bf16_t><<<grid, 256, 0, s>>>((const bf16_t *)w_packed, (bf16_t *const *)w_refs_dev, d, F, clt_pitch(d, 2));
    else k_unpack_vec<float><<<grid, 256, 0, s>>>((const float *)w_packed, (float *const *)w_refs_dev, d, F, clt_pitch(d, 4));
  } else {
    if (dtype != CLT_F32) k_unpack<bf16_t><<<grid, 256, 0, s>>>((const bf16_t *)w_packed, (bf16_t *const *)w_refs_dev, d, F, clt_pitch(d, 2));
    else k_unpack<float><<<grid, 256, 0, s>>>((const float *)w_packed, (float *const *)w_refs_dev, d, F, clt_pitch(d, 4));
  }
  return clt_check_launch();
}

extern "C" int clt_densify(const int32_t *row_ptr, const int32_t *col, const void *val, void *out, int64_t T,
                           int64_t F, int64_t L, int64_t out_layer_stride, int dtype, int out_f32, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T < 0 || F < 0 || L <= 0) return CLT_ERR_ARG;
  if (T == 0 || F == 0) return CLT_OK;
  if (!row_ptr || !out) return CLT_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const int64_t oe = dtype == CLT_F32 || out_f32 ? 4 : 2, pieces = clt_ceil_div(F * oe, DENSIFY_BYTES);
  if (F * oe % 16 == 0 && out_layer_stride * oe % 16 == 0 && clt_aligned16(out) && L * T * pieces <= 0x7FFFFFFFll) {
    const unsigned blocks = (unsigned)(L * T * pieces);
#define CLT_DENSIFY(TT, OT) \
  k_densify_rows<TT, OT><<<blocks, 256, 0, s>>>(row_ptr, col, (const TT *)val, (OT *)out, T, F, (int)pieces, out_layer_stride)
    if (dtype == CLT_F32) CLT_DENSIFY(float, float);
    else if (out_f32 && dtype == CLT_F16) CLT_DENSIFY(f16_t, float);
    else if (out_f32) CLT_DENSIFY(bf16_t, float);
    else CLT_DENSIFY(bf16_t, bf16_t);
#undef CLT_DENSIFY
    return clt_check_launch();
  }
  const int nb = 256 * 8;
  if (dtype == CLT_F32 || out_f32) k_zero_rows<float><<<nb, 256, 0, s>>>((float *)out, T, F, L, out_layer_stride);
  else k_zero_rows<bf16_t><<<nb, 256, 0, s>>>((bf16_t *)out, T, F, L, out_layer_stride);
  if (dtype == CLT_F32) k_densify_scatter<float, float><<<nb, 256, 0, s>>>(row_ptr, col, (const float *)val, (float *)out, T, F, L, out_layer_stride);
  else if (out_f32 && dtype == CLT_F16) k_densify_scatter<f16_t, float><<<nb, 256, 0, s>>>(row_ptr, col, (const f16_t *)val, (float *)out, T, F, L, out_layer_stride);
  else if (out_f32) k_densify_scatter<bf16_t, float><<<nb, 256, 0, s>>>(row_ptr, col, (const bf16_t *)val, (float *)out, T, F, L, out_layer_stride);
  else k_densify_scatter<bf16_t, bf16_t><<<nb, 256, 0, s>>>(row_ptr, col, (const bf16_t *)val, (bf16_t *)out, T, F, L, out_layer_stride);
  return clt_check_launch();
}

extern "C" int clt_decoder_norms(const void *w_packed, void *norms, int64_t d, int64_t F, int64_t L, int tying,
                                 int dtype, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (d <= 0 || F <= 0 || L <= 0 || tying < 0 || tying > 2 || !w_packed || !norms) return CLT_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == CLT_BF16) k_norms<bf16_t><<<256 * 8, 256, 0, s>>>((const bf16_t *)w_packed, (bf16_t *)norms, d, F, L, tying, clt_pitch(d, 2));
  else if (dtype == CLT_F16) k_norms<f16_t><<<256 * 8, 256, 0, s>>>((const f16_t *)w_packed, (f16_t *)norms, d, F, L, tying, clt_pitch(d, 2));
  else k_norms<float><<<256 * 8, 256, 0, s>>>((const float *)w_packed, (float *)norms, d, F, L, tying, clt_pitch(d, 4));
  return clt_check_launch();
}

extern "C" int clt_decode_route(int64_t T, int64_t d, int64_t F, int64_t L, int tying, int dtype,
                                size_t workspace_bytes) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T <= 0 || d <= 0 || F <= 0 || L <= 0 || L > 64 || tying < 0 || tying > 2) return CLT_ERR_ARG;
  return plan_route(d, F, tying, clt_elem_bytes(dtype), workspace_bytes >= decode_ws_bytes(T, d, L), true);
}

extern "C" int64_t clt_decoder_pitch(int64_t d, int dtype) {
  if (d <= 0 || !clt_model_dtype(dtype)) return -1;
  return clt_pitch(d, clt_elem_bytes(dtype));
}

extern "C" int64_t clt_decoder_slab_elems(int64_t d, int64_t F, int64_t L, int tying, int dtype) {
  if (d <= 0 || F <= 0 || L <= 0 || tying < 0 || tying > 2 || !clt_model_dtype(dtype)) return -1;
  const int64_t pitch = clt_pitch(d, clt_elem_bytes(dtype));
  const int64_t n_dec = tying == CLT_TYING_NONE ? L * (L + 1) / 2 : L;
  // the last element any schedule can touch: row F-1 of slot n_dec-1, formed like the kernels form it
  const int64_t last = decoder_slot_host(tying, L - 1, L - 1, L) * F * pitch + (F - 1) * pitch + (d - 1);
  return last + 1 == n_dec * F * pitch - (pitch - d) ? n_dec * F * pitch : -1;
}

extern "C" int clt_accumulate_dense(const int32_t *row_ptr, const int32_t *col, const void *val,
                                    const void *feat_offset, const void *feat_scale, void *acc, int64_t T,
                                    int64_t F, int64_t layer, int init, int dtype, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T < 0 || F <= 0 || (layer < 0 && !init)) return CLT_ERR_ARG;
  if (T == 0) return CLT_OK;
  if (!acc || (layer >= 0 && !row_ptr)) return CLT_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const unsigned nb = (unsigned)(clt_ceil_div(T, 4) < 8192 ? clt_ceil_div(T, 4) : 8192);
  if (init) {
    const int64_t bytes = T * F * (dtype != CLT_F32 ? 2 : 4);
    if (bytes % 16 == 0 && clt_aligned16(acc)) k_zero_quads<<<2048, 256, 0, s>>>((uint4 *)acc, bytes / 16);
    else if (dtype != CLT_F32) k_zero_rows<bf16_t><<<2048, 256, 0, s>>>((bf16_t *)acc, T, F, 1, T * F);
    else k_zero_rows<float><<<2048, 256, 0, s>>>((float *)acc, T, F, 1, T * F);
  }
  if (layer < 0) return clt_check_launch();   // clear only
  if (dtype == CLT_BF16)
    k_accumulate_dense<bf16_t><<<nb, 256, 0, s>>>(row_ptr, col, (const bf16_t *)val, (const bf16_t *)feat_offset,
                                                 (const bf16_t *)feat_scale, (bf16_t *)acc, T, F, layer, init);
  else if (dtype == CLT_F16)
    k_accumulate_dense<f16_t><<<nb, 256, 0, s>>>(row_ptr, col, (const f16_t *)val, (const f16_t *)feat_offset,
                                                 (const f16_t *)feat_scale, (f16_t *)acc, T, F, layer, init);
  else
    k_accumulate_dense<float><<<nb, 256, 0, s>>>(row_ptr, col, (const float *)val, (const float *)feat_offset,
                                                (const float *)feat_scale, (float *)acc, T, F, layer, init);
  return clt_check_launch();
}
