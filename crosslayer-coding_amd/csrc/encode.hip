// Encoder projection  pre[l] = x[l] . W[l]^T + b[l]   (reference clt/models/parallel.py:286)
//
// MFMA kernel for gfx950.  Both operands are K-contiguous (x is [T][d], W is [F][d]), so
// one loader serves both.
//
//   block tile  256 tokens x 256 features, 8 wavefronts (4 x 2), wave tile 64 x 128:
//               128 fp32 accumulators per lane, two wavefronts per SIMD, one block per CU
//   k step      128 bytes of K per LDS stage (64 bf16 / 32 fp32), two stages of 64 KB
//   loads       global_load_lds_dwordx4: 16 bytes per lane straight into LDS, no staging
//               registers.  LDS rows are 128 bytes; chunk c of row r lives at chunk position
//               c ^ ((r >> 1) & 7), which the loader realises by permuting which global chunk
//               each lane fetches, so the 16-byte fragment reads of a wavefront spread over
//               all banks
//   math        the matrix-core "A" operand is the W tile and "B" the x tile, so a lane ends
//               up with 4 consecutive features of one token per accumulator group
//   bias        the accumulators start from the bias, so it is added in fp32 before the one rounding
//   epilogue    rounding, then the tile goes through LDS so that the stores are 16 bytes per lane
//               and 256 contiguous bytes per token
//   bf16        v_mfma_f32_16x16x32_bf16, fp32 accumulate, one rounding (v_cvt_pk_bf16_f32)
//   fp32        v_mfma_f32_16x16x4_f32
#include <type_traits>
#include "select_state.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int BM = 256;   // tokens per block
constexpr int BN = 256;   // features per block
constexpr int ROWB = 128; // bytes of K per LDS row
constexpr int STAGE = (BM + BN) * ROWB;  // bytes of one LDS stage
constexpr int NWAVES = 8;                // wavefronts per block (4 x 2, wave tile 64 tokens x 128 features): two per SIMD
constexpr int NTHREADS = NWAVES * 64;
constexpr int CAND_LIST = 512;           // candidates of one 32-token piece the collecting epilogue lists in LDS
constexpr int ENC_SN = 8;  // feature tiles x token tiles that one XCD works on at a time
constexpr int ENC_SM = 4;


template <typename T> struct Mma;
template <> struct Mma<bf16_t> {
  __device__ static __forceinline__ void run(f32x16_t &acc, const uint4 &a, const uint4 &b) {
    bf16x8_t av = __builtin_bit_cast(bf16x8_t, a), bv = __builtin_bit_cast(bf16x8_t, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
  }
};
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
template <> struct Mma<f16_t> {
  __device__ static __forceinline__ void run(f32x16_t &acc, const uint4 &a, const uint4 &b) {
    f16x8_t av = __builtin_bit_cast(f16x8_t, a), bv = __builtin_bit_cast(f16x8_t, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
  }
};
template <> struct Mma<float> {
  __device__ static __forceinline__ void run(f32x16_t &acc, const uint4 &a, const uint4 &b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.x), __uint_as_float(b.x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.y), __uint_as_float(b.y), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.z), __uint_as_float(b.z), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.w), __uint_as_float(b.w), acc, 0, 0, 0);
  }
};

// element j of a 16-byte slot as a float
template <typename T> __device__ __forceinline__ float slot_elem(const uint4 &w, int j);
template <> __device__ __forceinline__ float slot_elem<float>(const uint4 &w, int j) {
  return __uint_as_float(j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w);
}

// The same on 16 x 16 tiles, 64 bytes of K per row: what the 256 x 256 tiles are made of.  Under full load the part is held by
// its power limit, and this shape moves its accumulators half as often per product: a loop of nothing but matrix
// instructions on random bf16 operands runs at 2030 TFLOP/s with it and at 1806 with 32 x 32 x 16 (profiles/matrix_rates.txt).
template <typename T> struct Mma16;
template <> struct Mma16<bf16_t> {
  static constexpr int PARTS = 1;
  __device__ static __forceinline__ void run(f32x4_t &acc, const uint4 &a, const uint4 &b, int) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
  }
};
template <> struct Mma16<f16_t> {
  static constexpr int PARTS = 1;
  __device__ static __forceinline__ void run(f32x4_t &acc, const uint4 &a, const uint4 &b, int) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), acc, 0, 0, 0);
  }
};
template <> struct Mma16<float> {
  static constexpr int PARTS = 4;        // one instruction per element of the fragments
  __device__ static __forceinline__ void run(f32x4_t &acc, const uint4 &a, const uint4 &b, int part) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(slot_elem<float>(a, part), slot_elem<float>(b, part), acc, 0, 0, 0);
  }
};

// 16 or 4 bytes per lane from base + off (bytes) straight into LDS: lane i of the wavefront lands at lds_at + 16 i or 4 i
// (lds_at wave-uniform).  As statements the compiler does not count: it cannot tell which of the loads on their way an
// LDS read depends on and would wait for all of them in front of every fragment read.  The waits are written out by hand.
__device__ __forceinline__ uint32_t lds_address(const void *p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
__device__ __forceinline__ void fill16(const void *base, uint32_t off, uint32_t lds_at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"((const char *)base + off), "{m0}"(lds_at) : "memory");
}
__device__ __forceinline__ void fill4(const void *base, uint32_t off, uint32_t lds_at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"((const char *)base + off), "{m0}"(lds_at) : "memory");
}

typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;

// two fp32 -> packed 16-bit elements (round to nearest even; bf16: one v_cvt_pk_bf16_f32)
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
template <typename T> __device__ __forceinline__ uint32_t pack16x2(float a, float b) {
  f32x2_t v = {a, b};
  if constexpr (IsHalf<T>::value) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// the same of the 16-bit types
template <> __device__ __forceinline__ float slot_elem<bf16_t>(const uint4 &w, int j) {
  const uint32_t u = (j >> 1) == 0 ? w.x : (j >> 1) == 1 ? w.y : (j >> 1) == 2 ? w.z : w.w;
  return __uint_as_float((j & 1) ? (u & 0xFFFF0000u) : (u << 16));
}
template <> __device__ __forceinline__ float slot_elem<f16_t>(const uint4 &w, int j) {
  const uint32_t u = (j >> 1) == 0 ? w.x : (j >> 1) == 1 ? w.y : (j >> 1) == 2 ? w.z : w.w;
  return f16_bits_to_f32((j & 1) ? (u >> 16) : (u & 0xFFFFu));
}
// element j as raw bits
template <typename T> __device__ __forceinline__ uint32_t slot_raw(const uint4 &w, int j);
template <> __device__ __forceinline__ uint32_t slot_raw<float>(const uint4 &w, int j) {
  return j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w;
}
template <> __device__ __forceinline__ uint32_t slot_raw<bf16_t>(const uint4 &w, int j) {
  const uint32_t u = (j >> 1) == 0 ? w.x : (j >> 1) == 1 ? w.y : (j >> 1) == 2 ? w.z : w.w;
  return (j & 1) ? (u >> 16) : (u & 0xFFFFu);
}

template <> __device__ __forceinline__ uint32_t slot_raw<f16_t>(const uint4 &w, int j) { return slot_raw<bf16_t>(w, j); }

// packed 16-bit helpers (two elements per 32-bit word)
typedef short i16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_sub_sat16(uint32_t a, uint32_t b) {   // signed saturating a - b
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(i16x2_t, a), __builtin_bit_cast(i16x2_t, b)));
}
__device__ __forceinline__ uint32_t pk_sign16(uint32_t a) {                 // 0xFFFF where the half is negative
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(i16x2_t, a) >> (short)15);
}
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a), __builtin_bit_cast(u16x2_t, b)));
}

// inclusive prefix sums with DPP row shifts: inside each row of 16 lanes / over the wavefront
__device__ __forceinline__ uint32_t row16_inclusive_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  return v;
}
__device__ __forceinline__ uint32_t wave_inclusive_scan32(uint32_t v) {
  v = row16_inclusive_scan(v);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Requires K % (128 / sizeof(T)) == 0 (whole LDS stages), M >= BM and N >= BN.  A tile that
// would stick out of the matrix is shifted back inside (its overlap with the neighbour is
// computed twice and stored by the neighbour only), so no load is predicated.
//
// Block -> tile map: workgroups go to the 8 XCDs round-robin, so block b runs on XCD b % 8.
// When the feature tiles split evenly, XCD x takes the feature tiles n = x, x+8, ... in groups
// (see the map below): a W tile is fetched by one XCD only.
//
// COLLECT 0 stores the tile.  COLLECT 1 / 2 store nothing: the epilogue compares every element
// with the layer's cut value (1) or its feature's threshold (2) and appends the ones that reach
// it, as (feature, raw value) entries ordered by (token, feature), to one extent of the layer's
// candidate pool per wavefront and feature segment (see CollectArgs).  A tile that was shifted
// back, in either direction, reports only the tokens and features its neighbour does not own.
// SEG (storing mode only): K is made of segments of `sps` stages each; segment q of a row starts
// q * xss (x) / q * wss (W) elements after the row's first segment and rows are xrs / wrs elements apart,
// so both operands may be gathered from several matrices side by side (see clt_encode_segmented).
struct SegArgs {
  int sps;           // stages per segment
  uint32_t magic;    // ceil(2^32 / sps): segment of stage i = (i * magic) >> 32 for i < 2^16
  int64_t xss, wss;  // segment strides, elements
  int xrs, wrs;      // row strides, elements
};

template <typename T, int COLLECT, bool SEG, bool ODD>
__global__ __launch_bounds__(NTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_encode_mfma(
    const T *__restrict__ x, const T *__restrict__ w, const T *__restrict__ bias, T *__restrict__ pre,
    int M, int K, int N, int tiles_m, int tiles_n, int total_tiles, int64_t xs, int64_t wstr, int64_t bs,
    int64_t ps, const SelState *__restrict__ gate, CollectArgs ca, SegArgs sg, int by_tokens) {
  static_assert(!SEG || COLLECT == 0, "segmented operands only in the storing mode");
  static_assert(!SEG || !ODD, "segmented operands come in an even number of stages");
  constexpr int CE = 16 / (int)sizeof(T);  // elements per 16-byte chunk
  constexpr int BK = ROWB / (int)sizeof(T);
  // Persistent workgroups (the grid is one block per CU, block b takes the tiles b, b + gridDim.x, ...)
  // that overlap the start of the next tile with the end of this one: the epilogue parks only in the
  // second stage buffer, 32 tokens of a wave tile at a time, so the first stage of the next tile is asked
  // for during the last two stages of this one.
  //
  // What bounds it: the power limit (1.7 - 1.9 GHz under load) and, at K of a few hundred, the epilogue and the turn of the
  // tiles, which the matrix cores wait out.  Against 32 x 32 x 16 products with all loads of a stage asked for at one barrier
  // (one stage to arrive) and a wait for the epilogue's stores at the turn, ms, bf16:
  //   L 12, T 4096, d 768, F 24576   1.84 -> 1.66 (1117 TFLOP/s)      L 4, T 8192, d 2048, F 16384   1.82 -> 1.65 (1330)
  //   T 8192, d 16384, F 2048        0.453 -> 0.388 (1420)            T = d = F = 8192               0.852 -> 0.768 (1430)
  // The vendor library takes 0.377 and 0.67 ms for the d 16384 and the 8192 product.  float32 (L 12, T 1024, d 768, F 6144):
  // 0.915 ms both (and with 32 x 32 x 2 products in this pipeline, one barrier a stage: which sums over K in another order).  Measured and dropped: the two wavefronts of a SIMD taking turns at multiplying and reading (1.95
  // ms at the first shape: with 64 KB per stage also coming into LDS, the reads of a turn outlast the other's products).
  __shared__ __attribute__((aligned(16))) unsigned char stage0[STAGE];
  __shared__ __attribute__((aligned(16))) unsigned char stage1[STAGE];
  __shared__ uint16_t cand_list[COLLECT ? NWAVES : 1][COLLECT ? CAND_LIST : 1];   // per wavefront, see the emission
  __shared__ __attribute__((aligned(16))) T bias_lds[NWAVES][128];                // per wavefront: the bias of its features
  __shared__ __attribute__((aligned(16))) T theta_lds[2][COLLECT == 2 ? NWAVES : 1][COLLECT == 2 ? 128 : 8];   // and their thresholds, this tile's and the next one's
  __shared__ __attribute__((aligned(16))) uint32_t cut_lds[2][COLLECT == 1 ? NWAVES : 1][4];                // the layer's cut key, likewise

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;   // wave tile: tokens [64 wm, +64) x features [128 wn, +128)
  const int per_layer = tiles_m * tiles_n;
  // The K loop walks its stages in pairs.  An odd number of stages (ODD, a separate instantiation so that the
  // even case pays nothing for it) gets a repeat of the last one appended, which is loaded like any other (every
  // count the pipeline's waits rely on stays the same) and multiplied by nothing.
  const int nk_real = K / BK;
  constexpr bool odd = ODD;
  const int nk = nk_real + (odd ? 1 : 0);

  struct TileAt { int layer, tm, tn, m0, n0, om0, on0, rot; };
  auto locate = [&](int bid) {
    TileAt t;
    t.layer = bid / per_layer;
    bid -= t.layer * per_layer;
    if (by_tokens) {
      // The mirror image, for products whose token operand is the larger one (the dense decoder product
      // summed [T, F] x W[t] [d, F]: few feature tiles, many token tiles): XCD x owns the TOKEN tiles
      // m = x, x+8, ..., so the large operand is fetched by one XCD only and the small one by all.
      const int xcd = bid & 7, idx = bid >> 3, mloc = tiles_m >> 3;
      const int g = idx / (ENC_SN * tiles_n), r = idx - g * ENC_SN * tiles_n;
      const int cnt = (mloc - g * ENC_SN) < ENC_SN ? (mloc - g * ENC_SN) : ENC_SN;
      const int ng = r / (cnt * ENC_SM), r2 = r - ng * cnt * ENC_SM;
      t.tn = ng * ENC_SM + r2 / cnt;
      t.tm = (g * ENC_SN + r2 % cnt) * 8 + xcd;
    } else if ((tiles_n & 7) == 0) {
      // XCD x owns the feature tiles n = x, x+8, ...  Its tiles run in groups of ENC_SN feature tiles
      // x ENC_SM token tiles (about one tile per CU of the XCD): the group's W tiles stay in the L2
      // while the token groups sweep past, so W is fetched once and the x slab once per ENC_SN tiles.
      const int xcd = bid & 7, idx = bid >> 3, nloc = tiles_n >> 3;
      const int g = idx / (ENC_SN * tiles_m), r = idx - g * ENC_SN * tiles_m;
      const int cnt = (nloc - g * ENC_SN) < ENC_SN ? (nloc - g * ENC_SN) : ENC_SN;
      const int mg = r / (cnt * ENC_SM), r2 = r - mg * cnt * ENC_SM;
      t.tm = mg * ENC_SM + r2 / cnt;
      t.tn = (g * ENC_SN + r2 % cnt) * 8 + xcd;
    } else {
      t.tn = bid / tiles_m; t.tm = bid - t.tn * tiles_m;
    }
    t.m0 = t.tm * BM; t.n0 = t.tn * BN;
    t.om0 = t.m0; t.on0 = t.n0;       // what the tile owns: it stores nothing before these
    if (t.m0 + BM > M) t.m0 = M - BM;
    if (t.n0 + BN > N) t.n0 = N - BN;
    // K is walked from a tile-dependent starting stage, wrapping around: the CUs of an XCD that share an
    // x tile or a W tile then ask for different lines of it at any one time, so one of them takes the
    // L2 miss and the others find the line there later, instead of all of them queueing behind the miss.
    // (no rotation with an appended stage: that one must come last)
    t.rot = odd ? 0 : (by_tokens ? 3 * t.tn + (t.tm >> 3) : (tiles_n & 7) == 0 ? 3 * t.tm + (t.tn >> 3) : t.tm + t.tn) % nk;
    return t;
  };
  // the storing mode computes only the layers that asked for it when a gate is given; the states of up to
  // 64 layers are fetched with one load
  const int nlayer = total_tiles / per_layer;
  unsigned long long want_mask = ~0ull;
  if (COLLECT == 0 && gate && nlayer <= 64)
    want_mask = __ballot(lane < nlayer && gate[lane < nlayer ? lane : 0].status == ST_RETRY);
  auto wanted = [&](int bid) {
    if (COLLECT != 0 || !gate) return true;
    const int l = bid / per_layer;
    return nlayer <= 64 ? ((want_mask >> l) & 1ull) != 0ull : gate[l].status == ST_RETRY;
  };
  if (COLLECT == 0 && gate && nlayer <= 64 && want_mask == 0ull) return;
  int bid = blockIdx.x;
  while (bid < total_tiles && !wanted(bid)) bid += gridDim.x;
  if (bid >= total_tiles) return;

  // ---- loader.  Per stage a wavefront brings in four 8-row groups of the x tile (rows 32 * wave + 8 t) and one of each
  // quarter j of the W tile (rows 128 * (wave / 4) + 32 j + 8 * (wave % 4)), 1 KB per instruction.  Lane l lands at row
  // l>>3, chunk position l&7 of its group and therefore fetches global chunk (l&7) ^ ((row >> 1) & 7).
  const int lr = lane >> 3, lp = lane & 7;
  const int xrs = SEG ? sg.xrs : K, wrs = SEG ? sg.wrs : K;     // row strides
  const uint32_t chE = (uint32_t)(lp ^ (lane >> 4)) * 16u;          // 8-row groups starting at a multiple of 16
  const uint32_t chO = (uint32_t)(lp ^ ((lane >> 4) | 4)) * 16u;    // ... at 8 mod 16
  const uint32_t xoffE = (uint32_t)lr * (uint32_t)xrs * (uint32_t)sizeof(T) + chE, xoffO = xoffE - chE + chO;
  const uint32_t woff = (uint32_t)lr * (uint32_t)wrs * (uint32_t)sizeof(T) + ((wave & 1) ? chO : chE);
  auto x_rows = [&](const TileAt &t) { return (const char *)(x + (int64_t)t.layer * xs + (int64_t)(t.m0 + wave * 32) * xrs); };
  auto w_rows = [&](const TileAt &t) {
    return (const char *)(w + (int64_t)t.layer * wstr + (int64_t)(t.n0 + (wave >> 2) * 128 + (wave & 3) * 8) * wrs);
  };
  // the stage walked kt-th by a tile (an index into K / BK)
  auto stage_k0 = [&](const TileAt &t, int kt) {
    int q = kt + t.rot;
    if (q >= nk) q -= nk;
    if constexpr (ODD) return q < nk_real ? q : nk_real - 1;
    return q;
  };
  // the i-th of a stage's eight loads: 8-row groups 0 - 3 of x, then W's quarters
  auto issue = [&](unsigned char *stage, const char *xt, const char *wt, int kst, int i) {
    int64_t xk = (int64_t)kst * BK, wk = xk;
    if constexpr (SEG) {
      const int q = sg.sps == 1 ? kst : (int)__umulhi((uint32_t)kst, sg.magic);
      const int kin = (kst - q * sg.sps) * BK;
      xk = q * sg.xss + kin;
      wk = q * sg.wss + kin;
    }
    if (i < 4) fill16(xt + ((int64_t)(i * 8) * xrs + xk) * (int64_t)sizeof(T), (i & 1) ? xoffO : xoffE,
                      lds_address(stage) + (wave * 32 + i * 8) * ROWB);
    else fill16(wt + ((int64_t)((i - 4) * 32) * wrs + wk) * (int64_t)sizeof(T), woff,
                lds_address(stage) + (BM + (wave >> 2) * 128 + (i - 4) * 32 + (wave & 3) * 8) * ROWB);
  };

  // ---- fragment reader: row l15 of each 16-row group; chunk (ks*4 + lq) at its swizzled position
  const int l15 = lane & 15, lq = lane >> 4;
  const int xrow = (wm * 64 + l15) * ROWB;              // + i * 16 * ROWB
  const int wrow = BM * ROWB + (wn * 128 + l15) * ROWB; // + j * 16 * ROWB
  int koff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) koff[ks] = ((ks * 4 + lq) ^ ((l15 >> 1) & 7)) << 4;

  // The accumulators start from the bias (the matrix core adds its products onto them in fp32), so
  // the epilogue has no bias loads or adds: accumulator (j, q) of a lane belongs to feature
  // j*16 + (lane>>4)*4 + q of the wave tile, whatever the token group i.  Each wavefront brings
  // the bias of its 128 features into LDS with one direct load ahead of the tile's stages - no register
  // holds it while the previous tile's epilogue runs - and reads it from there when the first stage has
  // landed.
  f32x4_t acc[4][8];
  constexpr int BIAS_LANES = 128 * (int)sizeof(T) / 16;   // lanes of the one 16-byte-per-lane load
  auto load_bias = [&](const TileAt &t, int slot) {
    if (bias && lane < BIAS_LANES) fill16(bias + (int64_t)t.layer * bs + t.n0 + wn * 128, lane * 16, lds_address(bias_lds[wave]));
    if constexpr (COLLECT == 2) {
      if (lane < BIAS_LANES)
        fill16((const T *)ca.theta + (int64_t)t.layer * ca.theta_stride + t.n0 + wn * 128, lane * 16, lds_address(theta_lds[slot][wave]));
    }
    // the layer's cut travels the same way: four bytes into the wavefront's slot, read in the epilogue
    if constexpr (COLLECT == 1) {
      if (lane == 0) fill4(&ca.st[t.layer].cut_key, 0, lds_address(cut_lds[slot][wave]));
    }
  };
  if (!bias && lane < BIAS_LANES)   // no bias: the slot holds zeros for good
    *reinterpret_cast<uint4 *>(reinterpret_cast<unsigned char *>(bias_lds[wave]) + lane * 16) = make_uint4(0u, 0u, 0u, 0u);
  // The bias is read with hand-written LDS loads and a hand-placed wait.
  const uint32_t bias_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)
                               reinterpret_cast<unsigned char *>(bias_lds[wave]) + (uint32_t)(lane >> 4) * 4u * (uint32_t)sizeof(T);
  auto init_acc = [&]() {
    typedef typename std::conditional<sizeof(T) == 4, uint4, uint2>::type braw_t;
    braw_t raw[8];
    // raw[j] = the 4 values at feature j * 16 of this lane's quarter.  All eight reads and their
    // wait are one statement, so no register is looked at before its value has arrived.
    if constexpr (sizeof(T) == 4) {
        asm volatile(
                     "ds_read_b128 %0, %8\n\t"
                     "ds_read_b128 %1, %8 offset:64\n\t"
                     "ds_read_b128 %2, %8 offset:128\n\t"
                     "ds_read_b128 %3, %8 offset:192\n\t"
                     "ds_read_b128 %4, %8 offset:256\n\t"
                     "ds_read_b128 %5, %8 offset:320\n\t"
                     "ds_read_b128 %6, %8 offset:384\n\t"
                     "ds_read_b128 %7, %8 offset:448\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(raw[0]), "=&v"(raw[1]), "=&v"(raw[2]), "=&v"(raw[3]), "=&v"(raw[4]), "=&v"(raw[5]), "=&v"(raw[6]), "=&v"(raw[7])
                     : "v"(bias_at));
    } else {
        asm volatile(
                     "ds_read_b64 %0, %8\n\t"
                     "ds_read_b64 %1, %8 offset:32\n\t"
                     "ds_read_b64 %2, %8 offset:64\n\t"
                     "ds_read_b64 %3, %8 offset:96\n\t"
                     "ds_read_b64 %4, %8 offset:128\n\t"
                     "ds_read_b64 %5, %8 offset:160\n\t"
                     "ds_read_b64 %6, %8 offset:192\n\t"
                     "ds_read_b64 %7, %8 offset:224\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(raw[0]), "=&v"(raw[1]), "=&v"(raw[2]), "=&v"(raw[3]), "=&v"(raw[4]), "=&v"(raw[5]), "=&v"(raw[6]), "=&v"(raw[7])
                     : "v"(bias_at));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float bv[4];
      if constexpr (sizeof(T) == 4) {
        bv[0] = __uint_as_float(raw[j].x); bv[1] = __uint_as_float(raw[j].y); bv[2] = __uint_as_float(raw[j].z); bv[3] = __uint_as_float(raw[j].w);
      } else {
        unpack_pair<T>(raw[j].x, bv[0], bv[1]);
        unpack_pair<T>(raw[j].y, bv[2], bv[3]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][j] = f32x4_t{bv[0], bv[1], bv[2], bv[3]};
    }
  };

  // Software pipeline over the K stages.  A stage is four quarters of 16 matrix operations: quarter q multiplies all of the
  // wavefront's tokens with 32 of its features (rows 32 q of the W half tile), over the stage's whole K.  The x fragments
  // stay in registers for the stage, each being replaced by the next stage's behind its last use; the W fragments of the next
  // quarter are read under this one's products.
  // Two barriers per stage, before the second and before the last quarter.  At the first, x and the first half of W have been
  // read by everybody, so six of the loads of the stage after next can be asked for, at the second the rest; and of the
  // stage's own loads, what the next two quarters read has landed: all of it but the last eight loads, so that a load has
  // a stage and a half to arrive.
  uint4 fx[4][2], fw[2][2][2];           // [token group][k-step], [buffer][feature group][k-step]
  auto read_x = [&](const unsigned char *st, int i, int ks) { fx[i][ks] = *reinterpret_cast<const uint4 *>(st + xrow + i * 16 * ROWB + koff[ks]); };
  auto read_w = [&](const unsigned char *st, int q, int j, int ks) {
    fw[q & 1][j][ks] = *reinterpret_cast<const uint4 *>(st + wrow + (q * 2 + j) * 16 * ROWB + koff[ks]);
  };
  auto meet = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  // `fresh`: the tile's first stage, all of which has landed before.
  // `first` / `rest`: ask for the i-th of the six / two loads into `st`.  `last`: the tile's last stage.
  // `m`: AND mask for the fragments of this stage (all ones, or zero for the appended stage, whose products must add nothing:
  // both operands are cleared, so that an infinity in the repeated data cannot turn into a NaN).
  auto body = [&](unsigned char *st, unsigned char *next, bool last, bool fresh, auto first, auto rest, uint32_t m) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q == 1 || q == 3) {
        if (q == 3 && last) __builtin_amdgcn_s_waitcnt(0xC07F);    // lgkmcnt(0)
        else if (q == 1 && fresh) __builtin_amdgcn_s_waitcnt(0xC07F);
        else __builtin_amdgcn_s_waitcnt(0x0078);                  // vmcnt(8) lgkmcnt(0)
        meet();
      }
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const int ks = g >> 2, i = g & 3;
#pragma unroll
        for (int part = 0; part < Mma16<T>::PARTS; ++part)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            uint4 xv = fx[i][ks], wv = fw[q & 1][j][ks];
            if constexpr (ODD) {
              xv.x &= m; xv.y &= m; xv.z &= m; xv.w &= m;
              wv.x &= m; wv.y &= m; wv.z &= m; wv.w &= m;
            }
            Mma16<T>::run(acc[i][q * 2 + j], wv, xv, part);
          }
        if (q < 3 && g < 4) read_w(st, q + 1, g & 1, g >> 1);
        if (q == 3 && !last) {
          if (g < 4) read_w(next, 0, g & 1, g >> 1);
          read_x(next, i, ks);
        }
        if (q == 0 && g == 1) rest(1);
        if ((q == 1 || q == 2) && g < 6 && (g & 1) == 0) first((q - 1) * 3 + g / 2);
        if (q == 3 && g == 1) rest(0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  TileAt cur = locate(bid);
  load_bias(cur, 0);
  {
    const int at = stage_k0(cur, 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) issue(stage0, x_rows(cur), w_rows(cur), at, i);
  }
  int slot = 0;
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0);
  meet();

  for (;;) {
    int nbid = bid + (int)gridDim.x;
    while (nbid < total_tiles && !wanted(nbid)) nbid += gridDim.x;
    const bool has_next = nbid < total_tiles;
    const TileAt nxt_tile = locate(has_next ? nbid : bid);
    const char *xt = x_rows(cur), *wt = w_rows(cur), *xn = x_rows(nxt_tile), *wn_ = w_rows(nxt_tile);
    const int m0 = cur.m0, n0 = cur.n0, layer = cur.layer;

    // here the first stage and the bias have landed for every wavefront, and the second buffer is free
    {
      const int at = stage_k0(cur, 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) issue(stage1, xt, wt, at, i);
    }
    init_acc();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) read_w(stage0, 0, j, ks);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) read_x(stage0, i, ks);
    int kt = 0;                           // nk is even
    for (; kt < nk - 2; kt += 2) {
      const int k1 = stage_k0(cur, kt + 1), k2 = stage_k0(cur, kt + 2), k3 = stage_k0(cur, kt + 3);
      body(stage0, stage1, false, kt == 0, [&](int i) { issue(stage0, xt, wt, k2, i); },
           [&](int i) { if (i == 0) issue(stage0, xt, wt, k2, 6); else if (kt > 0) issue(stage1, xt, wt, k1, 7); }, ~0u);
      body(stage1, stage0, false, false, [&](int i) { issue(stage1, xt, wt, k3, i); },
           [&](int i) { if (i == 0) issue(stage1, xt, wt, k3, 6); else issue(stage0, xt, wt, k2, 7); }, ~0u);
    }
    // the last two stages: the first buffer takes the next tile's first stage (at the end, one that nobody reads);
    // nothing may be on its way into the second one, which is parked in
    const int k1 = stage_k0(cur, kt + 1), k0 = stage_k0(nxt_tile, 0);
    body(stage0, stage1, false, kt == 0, [&](int i) { issue(stage0, xn, wn_, k0, i); },
         [&](int i) { if (i == 0) issue(stage0, xn, wn_, k0, 6); else if (kt > 0) issue(stage1, xt, wt, k1, 7); }, ~0u);
    body(stage1, stage0, true, false, [&](int i) { if (i == 0) load_bias(nxt_tile, slot ^ 1); },
         [&](int i) { if (i == 1) issue(stage0, xn, wn_, k0, 7); }, odd ? 0u : ~0u);
    // past the barrier of the last stage no wavefront reads either buffer any more

    // ---- epilogue.  The accumulator layout gives a lane 4 consecutive features of one token,
    // i.e. 8-byte pieces scattered over 32 rows per store - slow to write.  Each wavefront
    // therefore parks its tile in LDS, 32 tokens at a time (8 KB; two passes of 64 features for fp32) in its
    // eighth of the second stage buffer, and works on it row by row from there.
    // The next tile's first stage and its bias, asked for a stage ago, are waited for here: the stores that follow may then stay
    // under way into the next tile (loads and stores share a counter that runs in order).
    T *pl = pre + (int64_t)layer * ps;
    // The epilogue's addresses are rebuilt from the lane number for every tile.  Left visible as loop
    // invariants they would be computed once ahead of the tile loop and live across the K loop.
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int l31 = lane_e & 31, lh = lane_e >> 5, l15e = lane_e & 15, lqe = lane_e >> 4;
    unsigned char *park = stage1 + wave * (STAGE / 8);
    constexpr int NPASS = sizeof(T) == 2 ? 1 : 2;           // feature halves per pass
    constexpr int JP = 8 / NPASS;                            // 16-feature groups per pass
    // the 32 tokens h of feature pass `pass` -> rows of 256 bytes (128 bf16 / 64 fp32), 16-byte slots XOR-swizzled with
    // the row
    auto park_rows = [&](int pass, int h) {
#pragma unroll
      for (int jj = 0; jj < JP; ++jj) {
        const int j = pass * JP + jj;
        const int nl = jj * 16 + lqe * 4;                    // feature inside this pass
#pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
          const int ml = ii * 16 + l15e;                     // row inside the parked piece
          const f32x4_t y = acc[h * 2 + ii][j];
          if (sizeof(T) == 4) {
            const int slot = (nl >> 2) ^ (ml & 15);
            *reinterpret_cast<float4 *>(park + ml * 256 + slot * 16) = make_float4(y[0], y[1], y[2], y[3]);
          } else {
            const int slot = (nl >> 3) ^ (ml & 15);
            uint2 o;
            o.x = pack16x2<T>(y[0], y[1]);
            o.y = pack16x2<T>(y[2], y[3]);
            *reinterpret_cast<uint2 *>(park + ml * 256 + slot * 16 + (nl & 4) * 2) = o;
          }
        }
      }
    };
    constexpr int EPS = 16 / (int)sizeof(T);               // elements per 16-byte slot
#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) {
      if constexpr (COLLECT == 0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
        park_rows(pass, h);
        if (pass == 0 && h == 0) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), ahead of the stores
        // the wavefront reads its own piece back: lane -> (row = it*4 + lane/16, slot = lane%16)
#pragma unroll 4
        for (int it = 0; it < 8; ++it) {
          const int ml = it * 4 + (lane_e >> 4), sl = lane_e & 15;
          const uint4 v = *reinterpret_cast<const uint4 *>(park + ml * 256 + ((sl ^ (ml & 15)) * 16));
          const int m = m0 + wm * 64 + h * 32 + ml;
          const int n = n0 + wn * 128 + pass * (128 / NPASS) + sl * EPS;
          // the part of a shifted tile that its neighbour owns is left to the neighbour: the two walk K
          // from different stages, so their sums may differ in the last bit
          // (N is a multiple of 4, so a 16-byte piece of bf16 may straddle the line by half)
          if (m >= cur.om0) {
            if (n >= cur.on0) *reinterpret_cast<uint4 *>(pl + (int64_t)m * N + n) = v;
            else if (sizeof(T) == 2 && n + 4 >= cur.on0) *reinterpret_cast<uint2 *>(pl + (int64_t)m * N + n + 4) = make_uint2(v.z, v.w);
          }
        }
        }
      } else {
        // Two lanes per token row of the parked piece: lane -> row lane % 32, slots [8 hs, 8 hs + 8) with
        // hs = lane / 32.  Counting and ordering inside a half row need no cross-lane work; the two halves
        // of a row meet through one lane exchange.
        constexpr int KB = Elem<T>::KEYBITS;
        constexpr int SEGW = 128 / NPASS;                    // features per segment (16 slots)
        constexpr int NWL = SEGW / 64;                       // 32-bit mask words per lane (half a row)
        const int ncol0 = n0 + wn * 128 + pass * SEGW;       // first feature of the segment
        uint32_t cut_bits = 0;
        if constexpr (COLLECT == 1) {
          // The cut came in with the bias, during the tile before, and has long landed.  Read by hand, with its own wait
          // inside the statement: the compiler knows of no load that writes this slot.
          uint32_t cut_key_v;
          const uint32_t cut_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)cut_lds[slot][wave];
          asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(cut_key_v) : "v"(cut_at) : "memory");
          cut_bits = key_value_bits<T>((uint32_t)__builtin_amdgcn_readfirstlane((int)cut_key_v));
        }
        const bool cut_nan = (cut_bits & 0x7FFFFFFFu) > 0x7F800000u;   // only NaNs reach such a cut
        const float cutf = __uint_as_float(cut_bits);
        const int hs = lh, rsw = l31 & 15;
        const unsigned char *myrow = park + l31 * 256;
        uint32_t W[2][NWL];
        uint32_t cnt[2], part[2], incl[2], tot[2];           // own half row, the other half, rows up to this one
        // generic: float compares, element by element; bit c of a lane's mask = column 64 hs + c
        auto scan_generic = [&](uint32_t (&Wh)[NWL]) {
#pragma unroll
          for (int i = 0; i < NWL; ++i) Wh[i] = 0;
#pragma unroll
          for (int s8 = 0; s8 < 8; ++s8) {
            const int sl = hs * 8 + s8;
            const uint4 v = *reinterpret_cast<const uint4 *>(myrow + ((sl ^ rsw) * 16));
            uint4 tv = make_uint4(0, 0, 0, 0);
            if constexpr (COLLECT == 2)
              tv = *reinterpret_cast<const uint4 *>(theta_lds[slot][wave] + pass * SEGW + sl * EPS);
            uint32_t m = 0;
#pragma unroll
            for (int j = 0; j < EPS; ++j) {
              const float xv = slot_elem<T>(v, j);
              bool c;
              if constexpr (COLLECT == 1) c = cut_nan ? (xv != xv) : !(xv < cutf);
              else c = xv >= slot_elem<T>(tv, j);
              m |= (c ? 1u : 0u) << j;
            }
            Wh[(s8 * EPS) >> 5] |= m << ((s8 * EPS) & 31);
          }
        };
        // bf16 and a positive cut / threshold: x >= c  <=>  bits(x) >= bits(c) as signed 16-bit
        // integers (negative values have the sign bit), two elements per operation: the sign of
        // the saturated difference (c - 1) - x marks a candidate.  NaNs would be treated wrongly
        // (a top-k cut must take them all, also those with the sign bit set; a threshold must take
        // none), so the unsigned maximum of the raw values is tracked and the piece is redone with
        // float compares if it shows one.
        bool fast_ok = false;
        uint32_t cm1 = 0;
        const T *theta_seg = nullptr;
        if constexpr (sizeof(T) == 2) {
          if constexpr (COLLECT == 1) {
            const uint32_t cb = Elem<T>::raw(Elem<T>::from_f32(cutf));   // the cut is a value of T
            fast_ok = cb >= 1u && cb <= Elem<T>::INF16;
            cm1 = (cb - 1u) | ((cb - 1u) << 16);
          } else {
            theta_seg = theta_lds[slot][wave] + pass * SEGW;
            bool bad = false;
            if (lane_e < 16) {   // every threshold of the segment must be a positive number
              const uint4 tv = *reinterpret_cast<const uint4 *>(theta_seg + lane_e * 8);
              const uint32_t t4[4] = {tv.x, tv.y, tv.z, tv.w};
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                const uint32_t lo = t4[k] & 0xFFFFu, hi = t4[k] >> 16;
                bad = bad || lo < 1u || lo > Elem<T>::INF16 || hi < 1u || hi > Elem<T>::INF16;
              }
            }
            fast_ok = __ballot(bad) == 0;
          }
        }
        auto scan_piece = [&](uint32_t (&Wh)[NWL]) {
          bool done = false;
          if constexpr (sizeof(T) == 2) {
            if (fast_ok) {
              uint32_t mx = 0;
#pragma unroll
              for (int i = 0; i < NWL; ++i) Wh[i] = 0;
#pragma unroll
              for (int s8 = 0; s8 < 8; ++s8) {
                const int sl = hs * 8 + s8;
                const uint4 v = *reinterpret_cast<const uint4 *>(myrow + ((sl ^ rsw) * 16));
                const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
                uint32_t c4[4] = {cm1, cm1, cm1, cm1};
                if constexpr (COLLECT == 2) {
                  const uint4 tv = *reinterpret_cast<const uint4 *>(theta_seg + sl * 8);   // one address per half wave
                  c4[0] = tv.x - 0x00010001u; c4[1] = tv.y - 0x00010001u; c4[2] = tv.z - 0x00010001u; c4[3] = tv.w - 0x00010001u;
                }
                uint32_t a = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                  const uint32_t sg = pk_sign16(pk_sub_sat16(c4[k], w4[k]));   // 0xFFFF per candidate half
                  a |= sg & ((1u << (2 * k)) | (0x20000u << (2 * k)));         // element 2k -> bit 2k, 2k+1 -> bit 16+2k+1
                  mx = pk_max_u16(mx, COLLECT == 1 ? w4[k] : (w4[k] & 0x7FFF7FFFu));
                }
                const uint32_t m = (a | (a >> 16)) & 0xFFu;
                Wh[s8 >> 2] |= m << ((s8 & 3) * 8);
              }
              const uint32_t nan_above = COLLECT == 1 ? (0x8000u | Elem<T>::INF16) : Elem<T>::INF16;
              const bool nan_seen = (mx & 0xFFFFu) > nan_above || (mx >> 16) > nan_above;
              done = __ballot(nan_seen) == 0;
            }
          }
          if (!done) scan_generic(Wh);
        };
        uint2 *mypool = ca.pool + (unsigned long long)layer * ca.pool_cap;
        // Emission of the parked piece: `n` candidates, this lane's starting at position `first` of
        // the piece, to dst[0 .. n).  Each lane first drops a 16-bit code (row, column) for every
        // candidate of its half row into the wavefront's list, at the candidate's ordered position; then
        // the lanes take one candidate each: 64 consecutive pool entries per store instruction, and the
        // number of rounds is the piece's count / 64 instead of the fullest row's count.
        auto emit_piece = [&](const uint32_t (&Wh)[NWL], int h, uint32_t first, uint32_t n, uint2 *dst) {
          if (n <= (uint32_t)CAND_LIST) {
            uint16_t *lst = cand_list[wave];
            const uint32_t rowcode = ((uint32_t)l31 << 8) | (uint32_t)(hs * (SEGW / 2));
            uint32_t p = first;
#pragma unroll
            for (int i = 0; i < NWL; ++i) {
              uint32_t wd = Wh[i];
              while (wd) {
                lst[p++] = (uint16_t)(rowcode + (uint32_t)(i * 32 + (__ffs(wd) - 1)));
                wd &= wd - 1u;
              }
            }
#pragma unroll 2
            for (uint32_t idx = lane_e; idx < n; idx += 64) {
              const uint32_t code = lst[idx];
              const int ml = (int)(code >> 8), c = (int)(code & 255u);
              const int sl = c / EPS, j = c % EPS;
              const T rawv = *reinterpret_cast<const T *>(park + ml * 256 + ((sl ^ (ml & 15)) * 16) + j * (int)sizeof(T));
              dst[idx] = make_uint2(collect_place(h * 32 + ml, (uint32_t)(ncol0 + c)), Elem<T>::raw(rawv));
            }
          } else {
            // more candidates than the list holds: every lane walks its own half row
            uint32_t pos = first;
#pragma unroll
            for (int i = 0; i < NWL; ++i) {
              uint32_t wd = Wh[i];
              while (wd) {
                const int c = hs * (SEGW / 2) + i * 32 + (__ffs(wd) - 1);   // column inside the segment
                wd &= wd - 1u;
                const int sl = c / EPS, j = c % EPS;
                const T rawv = *reinterpret_cast<const T *>(myrow + ((sl ^ rsw) * 16) + j * (int)sizeof(T));
                dst[pos++] = make_uint2(collect_place(h * 32 + l31, (uint32_t)(ncol0 + c)), Elem<T>::raw(rawv));
              }
            }
          }
        };
        // the books are kept on the grid of whole tiles, in both directions: this wave tile's rows start at grid
        // row om0 + 64 wm, its segment is the one at feature on0 + 128 wn (+ the pass's half) of the grid
        const int nseg = tiles_n * BN / SEGW;
        const int seg = (cur.on0 + wn * 128 + pass * SEGW) / SEGW;
        const int Mp = tiles_m * BM, grow0 = cur.om0 + wm * 64;
        const int nrb = Mp / COLLECT_ROWS, rowblk = grow0 / COLLECT_ROWS;
        const int shift = cur.om0 - m0;                      // > 0: the tile was shifted back inside the matrix
        const int cshift = cur.on0 - ncol0;                  // > 0: the segment's first cshift features are the neighbour's
        const uint32_t tile = (uint32_t)seg * (uint32_t)nrb + (uint32_t)rowblk;
        uint32_t off = tile * ca.caps;                       // the tile's fixed slot
        // Each piece of 32 tokens is emitted into the fixed slot as soon as it is scanned, while it is
        // parked; the rare tile whose two pieces do not fit the slot takes an extent behind the slots (one
        // atomic) and parks and emits both again.
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          park_rows(pass, h);
          if (pass == 0 && h == 0) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), ahead of the stores
          scan_piece(W[h]);
          // the first `shift` tokens of a shifted tile belong to its neighbour, which reports them, and so do the
          // features in front of on0 (bit b of word i of a lane = feature hs * SEGW / 2 + 32 i + b of the segment)
          if (shift > 0 && wm * 64 + h * 32 + l31 < shift) {
#pragma unroll
            for (int i = 0; i < NWL; ++i) W[h][i] = 0;
          }
          if (cshift > 0) {
#pragma unroll
            for (int i = 0; i < NWL; ++i) {
              const int low = cshift - hs * (SEGW / 2) - i * 32;     // bits below `low` go
              W[h][i] &= low <= 0 ? ~0u : low >= 32 ? 0u : ~0u << low;
            }
          }
          cnt[h] = 0;
#pragma unroll
          for (int i = 0; i < NWL; ++i) cnt[h] += __popc(W[h][i]);
          part[h] = (uint32_t)__shfl_xor((int)cnt[h], 32);
          // rows up to and including this one, inside each half of the wavefront
          uint32_t v = row16_inclusive_scan(cnt[h] + part[h]);
          v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
          incl[h] = v;
          tot[h] = __builtin_amdgcn_readlane(v, 31);
          const uint32_t before = h ? tot[0] : 0u;
          const uint32_t first = incl[h] - cnt[h] - (hs ? 0u : part[h]);
          if (before + tot[h] <= ca.caps) emit_piece(W[h], h, first, tot[h], mypool + off + before);
        }
        const uint32_t total = tot[0] + tot[1];
        bool ok = true;
        if (total > ca.caps) {
          const unsigned long long fixed = (unsigned long long)nseg * nrb * ca.caps;
          uint32_t a = 0;
          if (lane_e == 0) a = atomicAdd(&ca.pool_count[layer], total);
          a = __builtin_amdgcn_readfirstlane(a);
          ok = fixed + a + total <= ca.pool_cap;
          off = (uint32_t)(fixed + a);
          if (!ok && lane_e == 0) atomicOr(&ca.st[layer].overflow, 1u);
          if (ok) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              park_rows(pass, h);
              emit_piece(W[h], h, incl[h] - cnt[h] - (hs ? 0u : part[h]), tot[h], mypool + off + (h ? tot[0] : 0u));
            }
          }
        }
        if (lane_e == 0) ca.tile_meta[(int64_t)layer * nseg * nrb + tile] = make_uint2(off, ok ? total : 0u);
      }
    }
    if (!has_next) break;
    // every wavefront is done with its parked rows before the next tile's loads overwrite them
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    meet();
    bid = nbid;
    cur = nxt_tile;
    slot ^= 1;
  }
  __builtin_amdgcn_s_waitcnt(0);   // no direct-to-LDS load may be in flight when the block retires
}

// ---- short batches ------------------------------------------------------------------------------------
// Fewer than BM tokens: the weights' one pass through the chip is the work, and a 256-token tile would multiply padding
// and leave most CUs idle on a small model (12 tiles at L = 3, F = 1024).  A block takes 32 NF features x 32 MT tokens;
// a stage is 128 bytes of K as above, and its four wavefronts split each stage's K between them - 32 K bytes each, so
// that even one block has four matrix cores at work - and add their sums through LDS at the end, in a fixed order.
// Three stages in LDS, two on their way: 30 - 72 KB in flight per CU, which is what HBM needs.
//
// Bound by the weights' HBM stream at few tokens (453 MB at L = 12, d = 768, F = 24576, bf16: 76 us for one token), by the
// blocks' repeated reads of x towards 128, and by the chain of K stages on a small model.  Against the 256-token tiles on
// a padded batch, us, at 1 / 32 / 77 / 128 / 255 tokens:
//   L 12, d 768, F 24576, bf16      76 / 94 / 141 / 176 / 303  against  178 / 186 / 189 / 200 / 228
//   L 16, d 2048, F 16384, bf16    197 / 206 / 266 / 309 / 549  against  334 / 335 / 337 / 346 / 382
//   L 12, d 768, F 6144, float32    46 / 44 / 108 / 143 / 251  against  385 / 380 / 385 / 388 / 402
//   L 3, d 768, F 1024, float32     13 / 12 / 14 / 18 / 18  against  184 / 185 / 187 / 188 / 189
// Hence the rule of encode_short_ok: up to 128 tokens (one block along them, W is read once), and up to 255 in float32,
// whose matrix products are what bounds, or where the large tiles would not fill the chip once.
constexpr int SK_STAGES = 3;

// As fill16, from a scalar base.
__device__ __forceinline__ void sk_fill16(const void *base, uint32_t off, uint32_t lds_at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds_at) : "memory");
}

template <typename T, int NF, int MT>
__global__ __launch_bounds__(256, 2) void k_encode_short(const T *__restrict__ x, const T *__restrict__ w, const T *__restrict__ bias,
                                                         T *__restrict__ pre, int M, int K, int N, int64_t xs, int64_t wstr,
                                                         int64_t bs, int64_t ps) {
  constexpr int WR = 32 * NF, XR = 32 * MT, BYTES = (WR + XR) * ROWB, LOADS = NF + MT;   // loads of a stage per wavefront
  constexpr int RP = WR + 4;                                // fp32 row pitch of the partial sums
  constexpr int RED = 4 * 32 * RP * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[SK_STAGES * BYTES > RED ? SK_STAGES * BYTES : RED];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * WR, m0 = blockIdx.y * XR, layer = blockIdx.z;
  const int nk = K * (int)sizeof(T) / ROWB;
  const char *wt = (const char *)(w + layer * wstr + (int64_t)n0 * K), *xt = (const char *)(x + layer * xs + (int64_t)m0 * K);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;

  // wavefront `wave` brings in the 8-row groups wave, wave + 4, ..: first those of W, then those of x.  Rows past the end
  // repeat the last one; nothing is stored for them.
  uint32_t off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (wave + 4 * (i < NF ? i : i - NF)) * 8 + (lane >> 3);
    const int left = i < NF ? N - n0 : M - m0;
    off[i] = (uint32_t)(r < left ? r : left - 1) * (uint32_t)K * (uint32_t)sizeof(T) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  auto issue = [&](int kt, uint32_t buf) {
    const uint32_t at = lds0 + buf * BYTES + (uint32_t)wave * 1024;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      sk_fill16((i < NF ? wt : xt) + (int64_t)kt * ROWB, off[i], at + (uint32_t)((i < NF ? i : i - NF) * 4096 + (i < NF ? 0 : WR * ROWB)));
  };

  f32x16_t acc[NF][MT];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[j][i][q] = 0.0f;
  const int l31 = lane & 31, lh = lane >> 5;
  const int frag = l31 * ROWB + (((wave * 2 + lh) ^ ((l31 >> 1) & 7)) << 4);      // this wavefront's quarter of a stage's K

  issue(0, 0);
  if (nk > 1) issue(1, 1);
  uint32_t buf = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // stage kt has landed (only the next one's loads may be under way), and this wavefront's reads of the stage before are over
    if (kt + 1 < nk) __builtin_amdgcn_s_waitcnt(0x0070 | LOADS);      // vmcnt(LOADS) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 2 < nk) issue(kt + 2, buf == 0 ? 2 : buf - 1);
    const unsigned char *st = lds + buf * BYTES + frag;
    uint4 fw[NF], fx[MT];
#pragma unroll
    for (int j = 0; j < NF; ++j) fw[j] = *reinterpret_cast<const uint4 *>(st + j * 32 * ROWB);
#pragma unroll
    for (int i = 0; i < MT; ++i) fx[i] = *reinterpret_cast<const uint4 *>(st + (WR + i * 32) * ROWB);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) Mma<T>::run(acc[j][i], fw[j], fx[i]);
    buf = buf == SK_STAGES - 1 ? 0 : buf + 1;
  }

  float *red = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    __syncthreads();                                        // the stages, or the tokens before these, have been read
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)
        *reinterpret_cast<float4 *>(red + (wave * 32 + l31) * RP + j * 32 + rg * 8 + lh * 4) =
            make_float4(acc[j][i][rg * 4], acc[j][i][rg * 4 + 1], acc[j][i][rg * 4 + 2], acc[j][i][rg * 4 + 3]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NF; ++u) {
      const int e = threadIdx.x + u * 256, tok = e / (WR / 4), c = e % (WR / 4) * 4;
      const int m = m0 + i * 32 + tok, n = n0 + c;
      if (m >= M || n >= N) continue;
      const float *p = red + tok * RP + c;
      float y[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float b = bias && n + q < N ? Elem<T>::to_f32(bias[layer * bs + n + q]) : 0.0f;
        y[q] = b + ((p[q] + p[32 * RP + q]) + (p[64 * RP + q] + p[96 * RP + q]));
      }
      T *o = pre + layer * ps + (int64_t)m * N + n;
      if ((N & 3) == 0) {                                   // whole quads, 8 or 16 bytes aligned (short_ok)
        if constexpr (sizeof(T) == 4) *reinterpret_cast<float4 *>(o) = make_float4(y[0], y[1], y[2], y[3]);
        else *reinterpret_cast<uint2 *>(o) = make_uint2(pack16x2<T>(y[0], y[1]), pack16x2<T>(y[2], y[3]));
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < N) o[q] = Elem<T>::from_f32(y[q]);
      }
    }
  }
}

// Any shape: one thread per output, fp32 accumulation.
template <typename T>
__global__ void k_encode_generic(const T *x, const T *w, const T *bias, T *pre, int64_t M, int64_t K, int64_t N,
                                 int64_t L, int64_t xs, int64_t wstr, int64_t bs, int64_t ps) {
  const int64_t total = M * N * L;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t l = i / (M * N), rem = i - l * M * N, m = rem / N, n = rem - m * N;
    const T *xr = x + l * xs + m * K, *wr = w + l * wstr + n * K;
    float acc = 0.0f;
    for (int64_t k = 0; k < K; ++k) acc = fmaf(Elem<T>::to_f32(xr[k]), Elem<T>::to_f32(wr[k]), acc);
    if (bias) acc += Elem<T>::to_f32(bias[l * bs + n]);
    pre[l * ps + m * N + n] = Elem<T>::from_f32(acc);
  }
}

template <typename T>
static bool encode_fast_ok(const void *x, const void *w, const void *b, const void *pre, int64_t T_, int64_t d,
                           int64_t F, int64_t xs, int64_t wstr, int64_t bs, int64_t ps) {
  constexpr int CE = 16 / (int)sizeof(T);
  return (d % (ROWB / (int)sizeof(T)) == 0) && (F % 4 == 0) && T_ >= BM && F >= BN && clt_aligned16(x) &&
         clt_aligned16(w) && clt_aligned16(pre) && (xs % CE == 0) && (wstr % CE == 0) && (ps % 4 == 0) &&
         (ps * (int64_t)sizeof(T)) % 16 == 0 && (F * (int64_t)sizeof(T)) % 8 == 0 && T_ < (1 << 30) &&
         F < (1 << 30) && d < (1 << 27) && (!b || (((uintptr_t)b) % 16 == 0 && bs % 8 == 0));
}

// What k_encode_short takes: a batch shorter than one tile (where it is the faster one, see there), whole 128-byte stages,
// aligned rows and output quads.
template <typename T>
static bool encode_short_ok(const void *x, const void *w, const void *pre, int64_t T_, int64_t d, int64_t F, int64_t L, int64_t xs,
                            int64_t wstr, int64_t ps) {
  constexpr int CE = 16 / (int)sizeof(T);
  const bool faster = T_ <= 128 || (T_ < BM && (sizeof(T) == 4 || clt_ceil_div(F, BN) * L <= 256));
  return faster && d % (ROWB / (int)sizeof(T)) == 0 && d < (1 << 22) && F < (1 << 30) && L <= 65535 && clt_aligned16(x) &&
         clt_aligned16(w) && clt_aligned16(pre) && xs % CE == 0 && wstr % CE == 0 && (F % 4 != 0 || ps % 4 == 0);
}

template <typename T>
static int launch_encode_short(const void *x, const void *w, const void *b, void *pre, int64_t T_, int64_t d, int64_t F, int64_t L,
                               int64_t xs, int64_t wstr, int64_t bs, int64_t ps, hipStream_t stream) {
  const int groups = (int)clt_ceil_div(T_, 32), ny = (int)clt_ceil_div(groups, 4), mt = (int)clt_ceil_div(groups, ny);
  // 64 features per block, which halves what is read of x, unless that leaves compute units idle
  const bool wide = clt_ceil_div(F, 64) * ny * L >= 256;
  const dim3 grid((unsigned)clt_ceil_div(F, wide ? 64 : 32), (unsigned)ny, (unsigned)L);
#define CLT_SHORT(NF, MT)                                                                                                  \
  k_encode_short<T, NF, MT><<<grid, 256, 0, stream>>>((const T *)x, (const T *)w, (const T *)b, (T *)pre, (int)T_, (int)d, \
                                                      (int)F, xs, wstr, bs, ps)
#define CLT_SHORT_MT(NF)                                                                                                   \
  switch (mt) { case 1: CLT_SHORT(NF, 1); break; case 2: CLT_SHORT(NF, 2); break; case 3: CLT_SHORT(NF, 3); break;         \
                default: CLT_SHORT(NF, 4); break; }
  if (wide) CLT_SHORT_MT(2) else CLT_SHORT_MT(1)
#undef CLT_SHORT_MT
#undef CLT_SHORT
  return clt_check_launch();
}

// One persistent workgroup per CU (a whole number of rounds over the 8 XCDs, so that block b stays on XCD
// b % 8 for all of its tiles), or one per tile when there are fewer tiles; 0 when the device cannot be asked.
static int64_t persistent_grid(int64_t tiles) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8)
    return 0;
  cus -= cus % 8;
  return tiles < cus ? tiles : cus;
}

template <typename T>
static int launch_encode(const void *x, const void *w, const void *b, void *pre, int64_t T_, int64_t d, int64_t F,
                         int64_t L, int64_t xs, int64_t wstr, int64_t bs, int64_t ps, int collect,
                         const SelState *gate, const CollectArgs *ca, hipStream_t stream) {
  const bool fast = encode_fast_ok<T>(x, w, b, collect ? nullptr : pre, T_, d, F, xs, wstr, bs, collect ? 16 : ps);
  if (collect && !fast) return CLT_ERR_ARG;
  if (!collect && encode_short_ok<T>(x, w, pre, T_, d, F, L, xs, wstr, ps))
    return launch_encode_short<T>(x, w, b, pre, T_, d, F, L, xs, wstr, bs, ps, stream);
  if (fast) {
    const int64_t tm = clt_ceil_div(T_, BM), tn = clt_ceil_div(F, BN);
    const int64_t nblk = tm * tn * L;
    if (nblk > 2147483647LL) return CLT_ERR_RANGE;
    CollectArgs none = {};
    const CollectArgs a = ca ? *ca : none;
    const int64_t grid = persistent_grid(nblk);
    if (grid <= 0) return CLT_ERR_LAUNCH;
    const SegArgs noseg = {};
    // which operand an XCD keeps to itself: the feature tiles (W, the larger one in the encoder), or the token
    // tiles when there are more of those and they split evenly over the XCDs
    const int by_tokens = (tm % 8 == 0 && tm > tn) ? 1 : 0;
#define CLT_ENC(C, O)                                                                                               \
  k_encode_mfma<T, C, false, O><<<(unsigned)grid, NTHREADS, 0, stream>>>((const T *)x, (const T *)w, (const T *)b,  \
                                                                     (T *)pre, (int)T_, (int)d, (int)F, (int)tm,  \
                                                                     (int)tn, (int)nblk, xs, wstr, bs, ps, gate,  \
                                                                     a, noseg, by_tokens)
    const bool odd_stages = ((d / (ROWB / (int64_t)sizeof(T))) & 1) != 0;
    if (odd_stages) {
      if (collect == 0) CLT_ENC(0, true);
      else if (collect == 1) CLT_ENC(1, true);
      else CLT_ENC(2, true);
    } else {
      if (collect == 0) CLT_ENC(0, false);
      else if (collect == 1) CLT_ENC(1, false);
      else CLT_ENC(2, false);
    }
#undef CLT_ENC
  } else {
    // the gate is ignored here: recomputing a layer that did not ask for it is harmless
    k_encode_generic<T><<<256 * 8, 256, 0, stream>>>((const T *)x, (const T *)w, (const T *)b, (T *)pre, T_, d, F, L,
                                                     xs, wstr, bs, ps);
  }
  return clt_check_launch();
}

// pre[T][F] = sum over segments q of x_q[T][dseg] . w_q[F][dseg]^T on the matrix-core kernel
template <typename T>
static int launch_encode_segmented(const void *x, const void *w, void *pre, int64_t T_, int64_t dseg, int64_t nseg,
                                   int64_t F, int64_t xss, int64_t xrs, int64_t wss, int64_t wrs, hipStream_t stream) {
  constexpr int CE = 16 / (int)sizeof(T);
  constexpr int BK = ROWB / (int)sizeof(T);
  const int64_t K = dseg * nseg;
  const bool ok = dseg % BK == 0 && (K / BK) % 2 == 0 && K / BK < 65536 && T_ >= BM && F >= BN && F % 4 == 0 &&
                  clt_aligned16(x) && clt_aligned16(w) && clt_aligned16(pre) && xss % CE == 0 && wss % CE == 0 &&
                  xrs % CE == 0 && wrs % CE == 0 && xrs < (1 << 24) && wrs < (1 << 24) && T_ < (1 << 30) &&
                  F < (1 << 30) && (F * (int64_t)sizeof(T)) % 8 == 0;
  if (!ok) return CLT_ERR_ARG;
  const int64_t tm = clt_ceil_div(T_, BM), tn = clt_ceil_div(F, BN), nblk = tm * tn;
  if (nblk > 2147483647LL) return CLT_ERR_RANGE;
  SegArgs sg;
  sg.sps = (int)(dseg / BK);
  sg.magic = (uint32_t)((0x100000000ull + (uint64_t)sg.sps - 1ull) / (uint64_t)sg.sps);
  sg.xss = xss; sg.wss = wss; sg.xrs = (int)xrs; sg.wrs = (int)wrs;
  const CollectArgs none = {};
  const int64_t grid = persistent_grid(nblk);
  if (grid <= 0) return CLT_ERR_LAUNCH;
  k_encode_mfma<T, 0, true, false><<<(unsigned)grid, NTHREADS, 0, stream>>>((const T *)x, (const T *)w, nullptr, (T *)pre, (int)T_,
                                                                    (int)K, (int)F, (int)tm, (int)tn, (int)nblk, 0, 0, 0,
                                                                    0, nullptr, none, sg, (tm % 8 == 0 && tm > tn) ? 1 : 0);
  return clt_check_launch();
}

}  // namespace

extern "C" int clt_encode_segmented(const void *x, const void *w, void *pre, int64_t T, int64_t d_seg, int64_t n_seg,
                                    int64_t F, int64_t x_seg_stride, int64_t x_row_stride, int64_t w_seg_stride,
                                    int64_t w_row_stride, int dtype, void *stream) {
  if (dtype != CLT_F32 && dtype != CLT_BF16) return CLT_ERR_DTYPE;
  if (T < 0 || d_seg <= 0 || n_seg <= 0 || F <= 0 || x_row_stride < d_seg || w_row_stride < d_seg || x_seg_stride < 0 ||
      w_seg_stride < 0)
    return CLT_ERR_ARG;
  if (T == 0) return CLT_OK;
  if (!x || !w || !pre) return CLT_ERR_ARG;
  if (dtype == CLT_BF16)
    return launch_encode_segmented<bf16_t>(x, w, pre, T, d_seg, n_seg, F, x_seg_stride, x_row_stride, w_seg_stride,
                                           w_row_stride, (hipStream_t)stream);
  return launch_encode_segmented<float>(x, w, pre, T, d_seg, n_seg, F, x_seg_stride, x_row_stride, w_seg_stride,
                                        w_row_stride, (hipStream_t)stream);
}

int clt_launch_encode(const void *x, const void *w, const void *b, void *pre, int64_t T, int64_t d, int64_t F,
                      int64_t L, int64_t xs, int64_t wstr, int64_t bs, int64_t ps, int dtype, int collect,
                      const SelState *gate, const CollectArgs *ca, hipStream_t stream) {
  if (dtype == CLT_BF16) return launch_encode<bf16_t>(x, w, b, pre, T, d, F, L, xs, wstr, bs, ps, collect, gate, ca, stream);
  if (dtype == CLT_F16) return launch_encode<f16_t>(x, w, b, pre, T, d, F, L, xs, wstr, bs, ps, collect, gate, ca, stream);
  return launch_encode<float>(x, w, b, pre, T, d, F, L, xs, wstr, bs, ps, collect, gate, ca, stream);
}

bool clt_encode_can_collect(const void *x, const void *w, const void *b, int64_t T, int64_t d, int64_t F,
                            int64_t xs, int64_t wstr, int64_t bs, int dtype) {
  const bool fast = dtype != CLT_F32 ? encode_fast_ok<bf16_t>(x, w, b, nullptr, T, d, F, xs, wstr, bs, 16)   // any 16-bit type
                                     : encode_fast_ok<float>(x, w, b, nullptr, T, d, F, xs, wstr, bs, 16);
  return fast && F <= (int64_t)COLLECT_COL + 1;
}

extern "C" int clt_encode_fast_path(const void *x, const void *w, const void *b, const void *pre, int64_t T, int64_t d,
                                    int64_t F, int64_t L, int64_t x_layer_stride, int64_t w_layer_stride,
                                    int64_t b_layer_stride, int64_t pre_layer_stride, int dtype) {
  if (!clt_model_dtype(dtype) || T <= 0 || d <= 0 || F <= 0 || L <= 0 || !x || !w || !pre) return 0;
  if (clt_ceil_div(T, BM) * clt_ceil_div(F, BN) * L > 2147483647LL) return 0;
  if (dtype != CLT_F32 ? encode_short_ok<bf16_t>(x, w, pre, T, d, F, L, x_layer_stride, w_layer_stride, pre_layer_stride)
                       : encode_short_ok<float>(x, w, pre, T, d, F, L, x_layer_stride, w_layer_stride, pre_layer_stride))
    return 1;
  const bool fast = dtype != CLT_F32
                        ? encode_fast_ok<bf16_t>(x, w, b, pre, T, d, F, x_layer_stride, w_layer_stride, b_layer_stride, pre_layer_stride)
                        : encode_fast_ok<float>(x, w, b, pre, T, d, F, x_layer_stride, w_layer_stride, b_layer_stride, pre_layer_stride);
  return fast ? 1 : 0;
}

extern "C" int clt_encode(const void *x, const void *w, const void *b, void *pre, int64_t T, int64_t d, int64_t F,
                          int64_t L, int64_t x_layer_stride, int64_t w_layer_stride, int64_t b_layer_stride,
                          int64_t pre_layer_stride, int dtype, void *stream) {
  if (!clt_model_dtype(dtype)) return CLT_ERR_DTYPE;
  if (T < 0 || d <= 0 || F <= 0 || L <= 0) return CLT_ERR_ARG;
  if (T == 0) return CLT_OK;
  if (!x || !w || !pre) return CLT_ERR_ARG;
  return clt_launch_encode(x, w, b, pre, T, d, F, L, x_layer_stride, w_layer_stride, b_layer_stride,
                           pre_layer_stride, dtype, 0, nullptr, nullptr, (hipStream_t)stream);
}

