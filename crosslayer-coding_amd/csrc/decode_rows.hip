// Sparse cross-layer decode of float32 models (reference clt/models/decoder.py:176-340) from LDS tiles: the gather of
// decode.hip is bound by the lines an L1 keeps outstanding, LDS hands rows out faster.
//
//   k_row_runs / k_row_streams / k_row_fill
//                   survivor list (CSR by token) -> one stream of records per group of 16 tokens, in the order in which
//                   k_decode_rows consumes them: by source, tile of SP_ROWS features, token
//   k_decode_rows   one workgroup per (target, 32 columns, part of the tokens): every tile of every source's decoder passes
//                   through LDS once, the sums stay in registers over all sources and features
//   k_grad_rows     the transposed product of the backward pass: decoder weight gradients from the same lists by feature,
//                   with the Adam step of the weights taken on the spot
#include "adam.h"
#include "spmm.h"

namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int DR_COLS = 32;                // columns of a tile: one 128-byte line
constexpr int DR_TOK = SP_GROUP;           // tokens of a wavefront: four accumulators per lane each
constexpr int DR_REC = 8;                  // entries of a record: a wavefront reads 8 rows x 16 bytes per lane
constexpr int DR_WAVES = 16;
constexpr int DR_QUAD = 4;                 // records of a slot
constexpr int DR_RING = 8;                 // slots that a wavefront keeps in LDS or on their way
constexpr int DR_LDS = 2 * SP_TILE_BYTES + DR_WAVES * DR_RING * 256;
constexpr int DR_THREADS = 256;
constexpr int DR_MAX_TILES = 512;
static_assert(DR_LDS <= 160 * 1024 && SP_ROWS / DR_REC <= 255, "record counts of a run are bytes");

// An entry: where its tile row begins in LDS (tile buffer and row), and its value.  A run - one token's entries of one tile -
// takes whole records; what is left of its last one repeats its last entry's place with value 0.  Four records of a stream lie
// together, the four that an eighth of a wavefront needs next to each other: two 16-byte reads bring them in.  Streams begin at
// whole quads.
__device__ __forceinline__ uint64_t dr_entry(uint64_t record, uint32_t e) {
  return record / DR_QUAD * (DR_QUAD * DR_REC) + e * DR_QUAD + record % DR_QUAD;
}
// A stream is a group's, over all layers - or, `by_layer`, a group's of one layer (number layer * groups + group).
struct RowPlan {
  int tiles, groups, parts, groups_per_part, stages, by_layer;        // stages: of a stream
  __device__ __forceinline__ int stream(int g, int s) const { return by_layer ? s * groups + g : g; }
  __device__ __forceinline__ int stage(int s, int c) const { return by_layer ? c : s * tiles + c; }
};

struct RunArgs {
  const int32_t *row_ptr, *col;
  const int32_t *src;      // the entry's value is val[src[j]]; null: val[j]
  const float *val;
  int64_t Tn, L, max_entries;      // what the records have room for: longer lists are left alone
  uint64_t layer_mask;
  RowPlan p;
  int32_t *start;          // [L * groups][DR_TOK][tiles + 1] list position where a token's entries of a tile begin
  uint4 *counts;           // [streams][stages] records per token, a byte each
  uint32_t *offset;        // [streams][stages] records of the stage, then of the stream before it
  uint32_t *total;         // [streams] records of the stream, in whole quads; by_layer: of the streams before it (k_row_firsts)
  uint2 *recs;
};

// One workgroup per (group of tokens, layer).  Rows are sorted by column, so a row's entries of one tile are a run, found by
// binary search.  A layer outside layer_mask counts as empty.
__global__ __launch_bounds__(DR_THREADS) void k_row_runs(RunArgs A) {
  extern __shared__ int32_t run_lds[];
  const int g = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, tiles = A.p.tiles;
  const int64_t tok0 = (int64_t)g * DR_TOK, r0 = (int64_t)s * A.Tn + tok0;
  const bool on = (A.layer_mask >> s) & 1ull;
  int32_t *out = A.start + ((int64_t)s * A.p.groups + g) * DR_TOK * (tiles + 1);
  for (int i = tid; i < DR_TOK * (tiles + 1); i += DR_THREADS) {
    const int tk = i / (tiles + 1), c = i - tk * (tiles + 1);
    int32_t lo = 0;
    if (on && tok0 + tk < A.Tn) {
      int32_t hi = A.row_ptr[r0 + tk + 1];
      lo = A.row_ptr[r0 + tk];
      const int32_t bound = c * SP_ROWS;
      if (c == tiles) lo = hi;
      while (lo < hi) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (A.col[mid] < bound) lo = mid + 1; else hi = mid;
      }
    }
    run_lds[i] = lo;
    out[i] = lo;
  }
  __syncthreads();
  for (int c = tid; c < tiles; c += DR_THREADS) {
    uint32_t w[4] = {0u, 0u, 0u, 0u}, sum = 0;
#pragma unroll
    for (int tk = 0; tk < DR_TOK; ++tk) {
      const uint32_t n = (uint32_t)(run_lds[tk * (tiles + 1) + c + 1] - run_lds[tk * (tiles + 1) + c] + DR_REC - 1) / DR_REC;
      w[tk >> 2] |= n << (8 * (tk & 3));
      sum += n;
    }
    const int64_t at = (int64_t)A.p.stream(g, s) * A.p.stages + A.p.stage(s, c);
    A.counts[at] = make_uint4(w[0], w[1], w[2], w[3]);
    A.offset[at] = sum;
  }
}

// One wavefront per stream: where each of its stages begins.
__global__ __launch_bounds__(64) void k_row_streams(RunArgs A) {
  const int lane = threadIdx.x;
  uint32_t *off = A.offset + (int64_t)blockIdx.x * A.p.stages;
  uint32_t run = 0;
  for (int st0 = 0; st0 < A.p.stages; st0 += 64) {
    const int st = st0 + lane;
    const uint32_t n = st < A.p.stages ? off[st] : 0u;
    uint32_t incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(incl, o);
      if (lane >= o) incl += up;
    }
    if (st < A.p.stages) off[st] = run + incl - n;
    run += __shfl(incl, 63);
  }
  if (lane == 0) A.total[blockIdx.x] = (run + DR_QUAD - 1) / DR_QUAD * DR_QUAD;
}

// Many streams: their totals become first records, by one workgroup.
constexpr int DR_FIRSTS = 1024;
__global__ __launch_bounds__(DR_FIRSTS) void k_row_firsts(uint32_t *total, int streams) {
  __shared__ uint32_t sums[DR_FIRSTS / 64];
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  uint32_t before = 0;
  for (int i0 = 0; i0 < streams; i0 += DR_FIRSTS) {
    const int i = i0 + threadIdx.x;
    const uint32_t n = i < streams ? total[i] : 0u;
    uint32_t incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(incl, o);
      if (lane >= o) incl += up;
    }
    if (lane == 63) sums[wave] = incl;
    __syncthreads();
    uint32_t mine = before, all = 0;
    for (int w = 0; w < DR_FIRSTS / 64; ++w) {
      mine += w < wave ? sums[w] : 0u;
      all += sums[w];
    }
    if (i < streams) total[i] = mine + incl - n;
    before += all;
    __syncthreads();
  }
}

// One workgroup per (group, layer): every run into its records.
__global__ __launch_bounds__(DR_THREADS) void k_row_fill(RunArgs A) {
  extern __shared__ int32_t fill_lds[];
  const int g = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, tiles = A.p.tiles, lane = tid & 63;
  if (A.row_ptr[A.L * A.Tn] > A.max_entries || !((A.layer_mask >> s) & 1ull)) return;
  int32_t *start = fill_lds;                               // [DR_TOK][tiles + 1]
  uint32_t *dest = (uint32_t *)(start + DR_TOK * (tiles + 1));      // [DR_TOK][tiles] first record of the run
  const int64_t tok0 = (int64_t)g * DR_TOK, r0 = (int64_t)s * A.Tn + tok0;
  const int32_t *src = A.start + ((int64_t)s * A.p.groups + g) * DR_TOK * (tiles + 1);
  for (int i = tid; i < DR_TOK * (tiles + 1); i += DR_THREADS) start[i] = src[i];
  const int stream = A.p.stream(g, s);
  const uint32_t base = A.p.by_layer ? A.total[stream] : stream_first(A.total, g, lane);
  const uint32_t stage0 = (uint32_t)(__popcll(A.layer_mask & ((1ull << s) - 1ull)) * tiles);
  __syncthreads();
  for (int c = tid; c < tiles; c += DR_THREADS) {
    uint32_t d = base + A.offset[(int64_t)stream * A.p.stages + A.p.stage(s, c)];
    for (int tk = 0; tk < DR_TOK; ++tk) {
      const int32_t b = start[tk * (tiles + 1) + c], n = start[tk * (tiles + 1) + c + 1] - b;
      dest[tk * tiles + c] = d;
      if (n % DR_REC != 0) {
        const uint32_t row = (uint32_t)(A.col[b + n - 1] - c * SP_ROWS);
        for (int i = n; i % DR_REC != 0; ++i) A.recs[dr_entry((uint64_t)d + i / DR_REC, i % DR_REC)] = make_uint2((((stage0 + c) & 1u) << 16) | (row << 7), 0u);
      }
      d += (uint32_t)(n + DR_REC - 1) / DR_REC;
    }
  }
  __syncthreads();
  for (int tk = tid >> 6; tk < DR_TOK; tk += DR_THREADS / 64) {
    if (tok0 + tk >= A.Tn) break;
    const int32_t e = A.row_ptr[r0 + tk + 1];
    for (int32_t j = A.row_ptr[r0 + tk] + lane; j < e; j += 64) {
      const int32_t f = A.col[j], c = f / SP_ROWS;
      const uint32_t i = (uint32_t)(j - start[tk * (tiles + 1) + c]);
      A.recs[dr_entry((uint64_t)dest[tk * tiles + c] + i / DR_REC, i % DR_REC)] =
          make_uint2((((stage0 + c) & 1u) << 16) | ((uint32_t)(f - c * SP_ROWS) << 7), __float_as_uint(A.val[A.src ? A.src[j] : j]));
    }
  }
}

struct RowArgs {
  RowPlan p;
  const uint4 *counts;
  const uint32_t *total;
  const uint2 *recs;
  const float *wp, *bias_sum, *skip_add;
  float *out;
  const int32_t *row_ptr, *col;
  const float *val;
  int64_t Tn, d, F, L, pitch, max_entries;
  uint64_t src_mask;
  int tying, t_begin, t_end, col_parts;
};

// ---- the records of one stage ---------------------------------------------------------------------------
// What a wavefront does between two barriers: the records of its 16 tokens that refer to the tile in LDS.  A record is one 16-byte
// read per lane (8 lanes a row, 8 rows) and four multiply-adds; the reads of the next two are under way while one is added.  In
// assembly, like the stages of spmm.h and for its reasons: there is code for every token and place of a record in two quads.
// Registers: v0 - v63 the sums (token k: v[4 k ..]), v64 - v79 four rows, v80 - v95 places and values of two quads of records, s[40:41]
// the next quad to ask for.  Behind the stage's last record two more are read in vain (their tile may still be on its way, and
// behind a stream's end they may be anything: a place is kept inside the tiles); the next stage begins by reading them again.
// Nothing is on its way into a register when the block ends.
typedef float dr_f32x32_t __attribute__((ext_vector_type(32)));
typedef uint32_t dr_u32x16_t __attribute__((ext_vector_type(16)));

// A row's place (bits 7 - 16) is put together with the lane's column by an exclusive choice of bits: the tiles begin at LDS address 0, where
// dynamic LDS lies as long as the kernels and what is inlined into them have no static __shared__ of their own.
#define DR_ROW(W, S) "v_and_or_b32 v96, " W ", %[inside], %[col]\n\tds_read_b128 v[" S "], v96\n\t"
// At places 0 and 4 the next quad is read (seven were asked for since that one, and the four loads of a tile if that is less than
// eight quads ago); two places later it has arrived, and its slot goes to the quad eight on.
#define DR_RING_READ(T, P, LO, HI)                                                              \
  "s_cmp_lt_i32 %[since], 8\n\t"                                                                \
  "s_cbranch_scc1 .Ldr_v" #T "_" #P "_%=\n\t"                                                   \
  "s_waitcnt vmcnt(7)\n"                                                                        \
  ".Ldr_v" #T "_" #P "_%=:\n\t"                                                                 \
  "s_waitcnt vmcnt(11)\n\t"                                                                     \
  "v_add_u32 v97, %[slot], %[ring_lane]\n\t"                                                    \
  "ds_read_b128 v[" LO "], v97\n\t"                                                             \
  "ds_read_b128 v[" HI "], v97 offset:16\n\t"
#define DR_RING_ASK                                                                             \
  "s_add_i32 m0, %[ring], %[slot]\n\t"                                                          \
  "s_add_i32 %[slot], %[slot], 0x100\n\t"                                                       \
  "global_load_lds_dword %[rec_lane], s[40:41]\n\t"                                             \
  "s_add_u32 s40, s40, 0x100\n\t"                                                               \
  "s_addc_u32 s41, s41, 0\n\t"                                                                  \
  "s_and_b32 %[slot], %[slot], 0x7ff\n\t"                                                       \
  "s_add_i32 %[since], %[since], 1\n\t"
#define DR_BOOKS_0(T) DR_RING_READ(T, 0, "88:91", "92:95")
#define DR_BOOKS_1(T)
#define DR_BOOKS_2(T) DR_RING_ASK
#define DR_BOOKS_3(T)
#define DR_BOOKS_4(T) DR_RING_READ(T, 4, "80:83", "84:87")
#define DR_BOOKS_5(T)
#define DR_BOOKS_6(T) DR_RING_ASK
#define DR_BOOKS_7(T)
// The record at place P of token T (sums A - D), and the one at place P + 2 with the word W, whose row goes to S; of the record's own
// row R0 - R3 and value V; BEHIND: reads under way behind the row's.
#define DR_CODE(T, A, B, C, D, P, N, W, S, V, R0, R1, R2, R3, BEHIND)                           \
  ".Ldr_b" #T "_" #P "_%=:\n\t"                                                                 \
  DR_BOOKS_##P(T) DR_ROW(W, S)                                                                  \
  "s_waitcnt lgkmcnt(" BEHIND ")\n\t"                                                           \
  "v_fmac_f32 " A ", " V ", " R0 "\n\t"                                                         \
  "v_fmac_f32 " B ", " V ", " R1 "\n\t"                                                         \
  "v_fmac_f32 " C ", " V ", " R2 "\n\t"                                                         \
  "v_fmac_f32 " D ", " V ", " R3 "\n\t"                                                         \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                 \
  "s_cbranch_scc1 .Ldr_x" #T "_" #N "_%=\n"
#define DR_TOKEN(T, A, B, C, D)                                                                 \
  DR_CODE(T, A, B, C, D, 0, 1, "v84", "72:75", "v81", "v64", "v65", "v66", "v67", "4")          \
  DR_CODE(T, A, B, C, D, 1, 2, "v86", "76:79", "v83", "v68", "v69", "v70", "v71", "2")          \
  DR_CODE(T, A, B, C, D, 2, 3, "v88", "64:67", "v85", "v72", "v73", "v74", "v75", "2")          \
  DR_CODE(T, A, B, C, D, 3, 4, "v90", "68:71", "v87", "v76", "v77", "v78", "v79", "2")          \
  DR_CODE(T, A, B, C, D, 4, 5, "v92", "72:75", "v89", "v64", "v65", "v66", "v67", "4")          \
  DR_CODE(T, A, B, C, D, 5, 6, "v94", "76:79", "v91", "v68", "v69", "v70", "v71", "2")          \
  DR_CODE(T, A, B, C, D, 6, 7, "v80", "64:67", "v93", "v72", "v73", "v74", "v75", "2")          \
  DR_CODE(T, A, B, C, D, 7, 0, "v82", "68:71", "v95", "v76", "v77", "v78", "v79", "2")          \
  "s_branch .Ldr_b" #T "_0_%=\n"
// behind token T, at place P: token N, whose number of records is COUNT (the subtraction borrows if there is none)
#define DR_SWITCH(T, N, COUNT, P)                                                               \
  ".Ldr_x" #T "_" #P "_%=:\n\t"                                                                 \
  "s_bfe_u32 %[n], " COUNT "\n\t"                                                               \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                 \
  "s_cbranch_scc0 .Ldr_b" #N "_" #P "_%=\n\t"                                                   \
  "s_branch .Ldr_x" #N "_" #P "_%=\n"
#define DR_SWITCHES(T, N, COUNT)                                                                \
  DR_SWITCH(T, N, COUNT, 0) DR_SWITCH(T, N, COUNT, 1) DR_SWITCH(T, N, COUNT, 2) DR_SWITCH(T, N, COUNT, 3) \
  DR_SWITCH(T, N, COUNT, 4) DR_SWITCH(T, N, COUNT, 5) DR_SWITCH(T, N, COUNT, 6) DR_SWITCH(T, N, COUNT, 7)
// four loads of the tile after this one, if there is one
#define DR_FILL(L)                                                                              \
  "s_mov_b32 %[since], 8\n\t"                                                                   \
  "s_cmp_eq_i32 %[to], -1\n\t"                                                                  \
  "s_cbranch_scc1 .Ldr_f" L "_%=\n\t"                                                           \
  "s_mov_b32 m0, %[to]\n\t"                                                                     \
  "s_mov_b32 %[since], 0\n\t"                                                                   \
  "global_load_lds_dwordx4 %[off0], %[from]\n\t"                                                \
  "s_add_i32 m0, %[to], 0x400\n\t"                                                              \
  "s_nop 0\n\t"                                                                                 \
  "global_load_lds_dwordx4 %[off1], %[from]\n\t"                                                \
  "s_add_i32 m0, %[to], 0x800\n\t"                                                              \
  "s_nop 0\n\t"                                                                                 \
  "global_load_lds_dwordx4 %[off2], %[from]\n\t"                                                \
  "s_add_i32 m0, %[to], 0xc00\n\t"                                                              \
  "s_nop 0\n\t"                                                                                 \
  "global_load_lds_dwordx4 %[off3], %[from]\n"                                                  \
  ".Ldr_f" L "_%=:\n\t"
// the stage's first two records, the first one at place P: their tile is there
#define DR_ENTER(P, W0, S0, W1, S1)                                                             \
  ".Ldr_e" #P "_%=:\n\t" DR_ROW(W0, S0) DR_ROW(W1, S1) DR_FILL(#P)                              \
  "s_bfe_u32 %[n], %[c0], 0x80000\n\t"                                                          \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                 \
  "s_cbranch_scc0 .Ldr_b0_" #P "_%=\n\t"                                                        \
  "s_branch .Ldr_x0_" #P "_%=\n"
#define DR_LAST(P) ".Ldr_x15_" #P "_%=:\n"
#define DR_STAGE                                                                                \
  "s_or_b32 %[n], %[c0], %[c1]\n\ts_or_b32 %[n], %[n], %[c2]\n\ts_or_b32 %[n], %[n], %[c3]\n\t" \
  "s_cmp_eq_u32 %[n], 0\n\ts_cbranch_scc1 .Ldr_none_%=\n\t"                                     \
  "s_bitcmp1_b32 %[at], 2\n\ts_cbranch_scc1 .Ldr_eb_%=\n\t"                                     \
  "s_bitcmp1_b32 %[at], 1\n\ts_cbranch_scc1 .Ldr_ea_%=\n\t"                                     \
  "s_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Ldr_e1_%=\n"                                       \
  DR_ENTER(0, "v80", "64:67", "v82", "68:71") DR_ENTER(1, "v82", "68:71", "v84", "72:75")       \
  ".Ldr_ea_%=:\n\ts_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Ldr_e3_%=\n"                        \
  DR_ENTER(2, "v84", "72:75", "v86", "76:79") DR_ENTER(3, "v86", "76:79", "v88", "64:67")       \
  ".Ldr_eb_%=:\n\ts_bitcmp1_b32 %[at], 1\n\ts_cbranch_scc1 .Ldr_ec_%=\n\t"                      \
  "s_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Ldr_e5_%=\n"                                       \
  DR_ENTER(4, "v88", "64:67", "v90", "68:71") DR_ENTER(5, "v90", "68:71", "v92", "72:75")       \
  ".Ldr_ec_%=:\n\ts_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Ldr_e7_%=\n"                        \
  DR_ENTER(6, "v92", "72:75", "v94", "76:79") DR_ENTER(7, "v94", "76:79", "v80", "64:67")       \
  DR_TOKEN(0, "v0", "v1", "v2", "v3") DR_SWITCHES(0, 1, "%[c0], 0x80008")                       \
  DR_TOKEN(1, "v4", "v5", "v6", "v7") DR_SWITCHES(1, 2, "%[c0], 0x80010")                       \
  DR_TOKEN(2, "v8", "v9", "v10", "v11") DR_SWITCHES(2, 3, "%[c0], 0x80018")                     \
  DR_TOKEN(3, "v12", "v13", "v14", "v15") DR_SWITCHES(3, 4, "%[c1], 0x80000")                   \
  DR_TOKEN(4, "v16", "v17", "v18", "v19") DR_SWITCHES(4, 5, "%[c1], 0x80008")                   \
  DR_TOKEN(5, "v20", "v21", "v22", "v23") DR_SWITCHES(5, 6, "%[c1], 0x80010")                   \
  DR_TOKEN(6, "v24", "v25", "v26", "v27") DR_SWITCHES(6, 7, "%[c1], 0x80018")                   \
  DR_TOKEN(7, "v28", "v29", "v30", "v31") DR_SWITCHES(7, 8, "%[c2], 0x80000")                   \
  DR_TOKEN(8, "v32", "v33", "v34", "v35") DR_SWITCHES(8, 9, "%[c2], 0x80008")                   \
  DR_TOKEN(9, "v36", "v37", "v38", "v39") DR_SWITCHES(9, 10, "%[c2], 0x80010")                  \
  DR_TOKEN(10, "v40", "v41", "v42", "v43") DR_SWITCHES(10, 11, "%[c2], 0x80018")                \
  DR_TOKEN(11, "v44", "v45", "v46", "v47") DR_SWITCHES(11, 12, "%[c3], 0x80000")                \
  DR_TOKEN(12, "v48", "v49", "v50", "v51") DR_SWITCHES(12, 13, "%[c3], 0x80008")                \
  DR_TOKEN(13, "v52", "v53", "v54", "v55") DR_SWITCHES(13, 14, "%[c3], 0x80010")                \
  DR_TOKEN(14, "v56", "v57", "v58", "v59") DR_SWITCHES(14, 15, "%[c3], 0x80018")                \
  DR_TOKEN(15, "v60", "v61", "v62", "v63")                                                      \
  ".Ldr_none_%=:\n\t" DR_FILL("n")                                                              \
  DR_LAST(0) DR_LAST(1) DR_LAST(2) DR_LAST(3) DR_LAST(4) DR_LAST(5) DR_LAST(6) DR_LAST(7)       \
  /* the tile's lines are waited for, not the quads asked for behind them; this wavefront's reads of the tile are over */ \
  "s_cmp_ge_i32 %[since], 8\n\ts_cbranch_scc1 .Ldr_8_%=\n\t"                                    \
  "s_cmp_ge_i32 %[since], 4\n\ts_cbranch_scc1 .Ldr_4_%=\n\t"                                    \
  "s_waitcnt vmcnt(0)\n"                                                                        \
  ".Ldr_4_%=:\n\ts_waitcnt vmcnt(4)\n"                                                          \
  ".Ldr_8_%=:\n\ts_waitcnt vmcnt(8) lgkmcnt(0)"

#define DR_STAGE_ASM(INSIDE, TILE, TO, OFF0, OFF1, OFF2, OFF3)                                                                       \
  asm volatile(DR_STAGE                                                                                                            \
               : "+{v[0:31]}"(lo), "+{v[32:63]}"(hi), "+{v[80:95]}"(words), "+{s[40:41]}"(next), [slot] "+s"(slot), [since] "=&s"(since), \
                 [n] "=&s"(n), "=&{m0}"(m0)                                                                                        \
               : [at] "s"(at), [c0] "s"(cnt.x), [c1] "s"(cnt.y), [c2] "s"(cnt.z), [c3] "s"(cnt.w), [ring] "s"(ring), [inside] "s"(INSIDE), \
                 [from] "s"(TILE), [to] "s"(TO), [off0] "v"(OFF0), [off1] "v"(OFF1), [off2] "v"(OFF2), [off3] "v"(OFF3), [col] "v"(col_lane), \
                 [ring_lane] "v"(ring_lane), [rec_lane] "v"(rec_lane)                                                              \
               : "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79", "v96", "v97", \
                 "scc", "memory")

// Two tiles of 512 features x 32 columns in LDS, one being read while the other comes in.  A wavefront owns 16 tokens; a
// record is one 16-byte read per lane (8 lanes a row, 8 rows) and four multiply-adds, its eight partial sums per column meet
// at the end.  The records come through a ring as in k_decode_tiles.  Workgroups that share a tile follow each other on one XCD.
//
// L = 12, d = 768, F = 6144, 1024 tokens, 200 survivors per token of which some have many more than others, untied: 1.44 ms (49 GB of
// gathered rows, 34 TB/s) against 2.62 ms of the gather from the L2s; 1.97 ms in loops over a token's records with the books of the
// ring in each step.  Bound by what LDS returns and by the number of a wavefront's instructions alike: 4.1 ns per record and CU for 1
// KB of rows and half as much of records, 10 instructions.
// Measured and dropped (in loops): the rows of the next record asked for ahead of the barrier (register moves); four records in one
// word per lane, handed out by DPP operands (bound by instruction issue).
__global__ __launch_bounds__(DR_WAVES * 64) void k_decode_rows(RowArgs A) {
  extern __shared__ __attribute__((aligned(128))) char tile_lds[];
  if (A.row_ptr[A.L * A.Tn] > A.max_entries) return;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int pair = (seq / A.p.parts) * 8 + xcd, part = seq % A.p.parts;
  if (pair >= (A.t_end - A.t_begin) * A.col_parts) return;
  const int t = A.t_end - 1 - pair / A.col_parts, cp = pair % A.col_parts;      // longest first
  const uint64_t mask = A.src_mask & ((2ull << t) - 1ull);
  const int n_stages = __popcll(mask) * A.p.tiles;
  const int g = part * A.p.groups_per_part + wave;
  const bool mine = wave < A.p.groups_per_part && g < A.p.groups;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)tile_lds;

  // this wavefront's share of a tile: 32 rows, eight at a time, 16 bytes per lane; rows past the matrix, which nobody refers to,
  // are read as its last one
  const uint32_t pitch_b = (uint32_t)(A.pitch * 4), col_b = (uint32_t)(lane & 7) * 16;
  const uint32_t off_a = (uint32_t)(wave * 32 + (lane >> 3)) * pitch_b + col_b;
  auto row_off = [&](int i, int rows) {
    const uint32_t off = off_a + (uint32_t)i * 8 * pitch_b, last = (uint32_t)((rows < SP_ROWS ? rows : SP_ROWS) - 1) * pitch_b + 112u;
    return off < last ? off : last;
  };
  auto tile_at = [&](int s) { return (const char *)A.wp + sp_slot(A.tying, s, t, A.L) * A.F * (int64_t)pitch_b + (int64_t)cp * 128; };

  dr_f32x32_t lo, hi;                                      // tokens 0 - 7 and 8 - 15
#pragma unroll
  for (int i = 0; i < 32; ++i) { lo[i] = 0.f; hi[i] = 0.f; }
  if (n_stages > 0) {
    const uint32_t ring = lds0 + 2 * SP_TILE_BYTES + (uint32_t)wave * (DR_RING * 256);
    const uint32_t rec_lane = (uint32_t)lane * 4, ring_lane = ring + (uint32_t)(lane >> 3) * 32, col_lane = lds0 + col_b;
    const char *quad = (const char *)(A.recs + (uint64_t)__builtin_amdgcn_readfirstlane(stream_first(A.total, mine ? g : 0, lane)) * DR_REC);
    auto ask = [&](uint32_t slot) {
      sp_fill4((const uint32_t *)quad, rec_lane, ring + slot);
      quad += 256;
    };
    uint64_t m = mask;
    int s = __ffsll((unsigned long long)m) - 1, c = 0, rows = (int)A.F;
    const char *tile = tile_at(s);
    const uint32_t lds_share = lds0 + (uint32_t)wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) sp_fill16(tile, row_off(i, rows), lds_share + (uint32_t)i * 1024);
#pragma unroll
    for (int i = 0; i < DR_RING; ++i) ask((uint32_t)i * 256);
    const auto stream_counts = (const __attribute__((address_space(4))) uint4 *)(uintptr_t)A.counts + (int64_t)(mine ? g : 0) * A.p.stages;
    auto count_at = [&](int at) {
      return mine ? make_uint4(stream_counts[at].x, stream_counts[at].y, stream_counts[at].z, stream_counts[at].w) : make_uint4(0u, 0u, 0u, 0u);
    };
    uint4 cnt = count_at(s * A.p.tiles);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the first quad's places and values: places 0 - 3 of eight; the next one's are read with the first record
    dr_u32x16_t words;
    {
      const auto q = (const __attribute__((address_space(3))) u32x4_t *)(uintptr_t)ring_lane;
      const u32x4_t a = q[0], b = q[1];
      words = __builtin_shufflevector(__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7), __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7),
                                      0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
      asm volatile("" ::"v"(words));                       // the slot has been read
      ask(0);
    }
    uint32_t slot = 256, at = 0;                           // of the next quad to read; place of the next record
    for (int st = 0; st < n_stages; ++st) {
      uint32_t to = SP_NO_TILE;                            // where this wavefront's share of the next tile goes, if there is one
      if (st + 1 < n_stages) {
        tile += SP_ROWS * pitch_b;
        rows -= SP_ROWS;
        if (++c == A.p.tiles) {
          c = 0;
          m &= m - 1;
          s = __ffsll((unsigned long long)m) - 1;
          tile = tile_at(s);
          rows = (int)A.F;
        }
        to = lds_share ^ (uint32_t)((st & 1) ^ 1) * SP_TILE_BYTES;
      }
      const uint4 cnt_next = count_at(s * A.p.tiles + c);
      const uint32_t off0 = row_off(0, rows), off1 = row_off(1, rows), off2 = row_off(2, rows), off3 = row_off(3, rows);
      asm volatile("" ::"v"(off0), "v"(off1), "v"(off2), "v"(off3) : "memory");
      __builtin_amdgcn_s_barrier();                        // tile st is complete, and nobody reads the other one any more
      asm volatile("" ::: "memory");
      uint32_t n, m0, since;
      at = __builtin_amdgcn_readfirstlane(at);             // (uniform, which the compiler does not see everywhere)
      slot = __builtin_amdgcn_readfirstlane(slot);
      uint64_t next = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)(uintptr_t)quad >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint64_t)(uintptr_t)quad);
      DR_STAGE_ASM(0x1FF80u, tile, to, off0, off1, off2, off3);
      quad = (const char *)(uintptr_t)next;
      // the stage's records, a byte per token (at most 64 each)
      const uint32_t even = (cnt.x & 0x00FF00FFu) + (cnt.y & 0x00FF00FFu) + (cnt.z & 0x00FF00FFu) + (cnt.w & 0x00FF00FFu);
      const uint32_t odd = ((cnt.x >> 8) & 0x00FF00FFu) + ((cnt.y >> 8) & 0x00FF00FFu) + ((cnt.z >> 8) & 0x00FF00FFu) + ((cnt.w >> 8) & 0x00FF00FFu);
      at += (even + odd) + ((even + odd) >> 16);           // (only its low three bits are looked at)
      cnt = cnt_next;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may be on its way into LDS when the workgroup ends
  }

  // lane 8 j + i holds entries j of every record, columns 4 i .. 4 i + 3: the eight sums meet in every lane, row tk is written
  // by lanes 8 (tk % 8) .. + 7
  auto meet = [&](f32x4v_t a) {
#pragma unroll
    for (int o = 8; o < 64; o <<= 1)
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] += __shfl_xor(a[q], o);
    return a;
  };
  const int64_t o = (int64_t)cp * DR_COLS + (lane & 7) * 4;
  auto write = [&](int tk, f32x4v_t a) {
    const int64_t tok = (int64_t)g * DR_TOK + tk;
    if (!mine || tok >= A.Tn || (lane >> 3) != (tk & 7)) return;
    const int64_t at = ((int64_t)t * A.Tn + tok) * A.d + o;
    if (A.bias_sum) a += *reinterpret_cast<const f32x4v_t *>(A.bias_sum + (int64_t)t * A.d + o);
    if (A.skip_add) a += *reinterpret_cast<const f32x4v_t *>(A.skip_add + at);
    *reinterpret_cast<f32x4v_t *>(A.out + at) = a;
  };
  uint32_t again = 0;                                      // tokens whose sums are not finite
#pragma unroll
  for (int tk = 0; tk < DR_TOK; ++tk) {
    f32x4v_t sum;
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] = tk < 8 ? lo[(tk & 7) * 4 + q] : hi[(tk & 7) * 4 + q];
    const f32x4v_t a = meet(sum);
    const float z = fmaf(a[0], 0.0f, fmaf(a[1], 0.0f, fmaf(a[2], 0.0f, a[3] * 0.0f)));
    if (ballot64(z != z) != 0) again |= 1u << tk;
    else write(tk, a);
  }
  // Those once more without the places that fill records up: 0 * inf of such a place would turn an infinity into a NaN.
  for (; again != 0; again &= again - 1) {
    const int tk = __ffs(again) - 1;
    f32x4v_t a{0.f, 0.f, 0.f, 0.f};
    for (uint64_t m = mask; m != 0; m &= m - 1) {
      const int s = __ffsll((unsigned long long)m) - 1;
      const float *w = A.wp + sp_slot(A.tying, s, t, A.L) * A.F * A.pitch + o;
      const int32_t *row = A.row_ptr + (int64_t)s * A.Tn + (int64_t)g * DR_TOK + tk;
      for (int32_t j = row[0] + (lane >> 3); j < row[1]; j += DR_REC) {
        const f32x4v_t x = *reinterpret_cast<const f32x4v_t *>(w + (int64_t)A.col[j] * A.pitch);
        const float v = A.val[j];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = fmaf(v, x[q], a[q]);
      }
    }
    write(tk, meet(a));
  }
}

// ---- decoder weight gradient and Adam -------------------------------------------------------------------
// dW[s->t][f][:] = sum over the tokens of feature f of value * g[t][token][:]: the same sums with features in the place of tokens
// - 16 features per wavefront, tiles of 512 tokens x 32 columns of g[t].
constexpr int GR_WAVES = 8;
constexpr int GR_LDS = SP_TILE_BYTES + GR_WAVES * DR_RING * 256;
static_assert(GR_LDS * 2 <= 160 * 1024, "two workgroups per CU");

struct GradRowArgs {
  RowPlan p;
  const uint4 *counts;
  const uint32_t *first;
  const uint2 *recs;
  const float *g;            // [L][T][d]
  float *w, *m, *v;          // packed decoders, moments
  const int32_t *list_ptr, *list_tok, *list_src;
  const float *val;
  int64_t Tn, d, F, L, pitch, max_entries;
  int64_t m_row, m_cols;     // moments: elements between rows and between column parts of eight
  int col_parts, items;      // items of one (source, target) pair per XCD
  AdamCoef adam;
};

// One workgroup per (source, target, 32 columns, 128 features).  Weights and moments stream through once (24 bytes per weight), in
// lines of 128 bytes: two workgroups share a CU (one tile buffer each), and one's sums run under the other's streaming.
//
// L = 12, d = 768, F = 6144, 1024 tokens, 200 survivors per token: 2.55 ms (8.8 GB of weights and moments, 3.4 TB/s), against 3.39 ms of 32-byte
// tiles and 0.57 ms for bringing those back into the slab; the training step 9.95 -> 8.76 ms.  Without entries 2.2 ms: what bounds it
// is the chain of a workgroup, tile, sums, tile, sums, moments, of which a CU has two under way.
__global__ __launch_bounds__(GR_WAVES * 64, 4) void k_grad_rows(GradRowArgs A) {
  extern __shared__ __attribute__((aligned(128))) char tile_lds[];
  if (A.list_ptr[A.L * A.F] > A.max_entries) return;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int slot_dec = seq / A.items, item = xcd * A.items + seq % A.items;
  if (item >= A.p.parts * A.col_parts) return;
  const int part = item / A.col_parts, cp = item % A.col_parts;
  int s = 0, t = slot_dec;                                 // decoder "0->0", "0->1", ..: source s, target t
  while (t >= (int)A.L - s) { t -= (int)A.L - s; ++s; }
  t += s;
  const int g = part * GR_WAVES + wave;
  const bool mine = g < A.p.groups;
  const int stream = s * A.p.groups + (mine ? g : 0);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)tile_lds;

  // this wavefront's share of a tile: 64 rows, eight at a time, 16 bytes per lane; rows past the batch are read as its last one
  const uint32_t pitch_b = (uint32_t)(A.d * 4), col_b = (uint32_t)(lane & 7) * 16;
  const char *tile = (const char *)A.g + (int64_t)t * A.Tn * (int64_t)pitch_b + (int64_t)cp * 128;
  auto fill = [&](int rows) {
    const uint32_t last = (uint32_t)((rows < SP_ROWS ? rows : SP_ROWS) - 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t row = (uint32_t)(wave * 64 + i * 8 + (lane >> 3));
      sp_fill16(tile, (row < last ? row : last) * pitch_b + col_b, lds0 + (uint32_t)(wave * 8192 + i * 1024));
    }
  };

  dr_f32x32_t lo, hi;                                      // features 0 - 7 and 8 - 15
#pragma unroll
  for (int i = 0; i < 32; ++i) { lo[i] = 0.f; hi[i] = 0.f; }
  {
    const uint32_t ring = lds0 + SP_TILE_BYTES + (uint32_t)wave * (DR_RING * 256);
    const uint32_t rec_lane = (uint32_t)lane * 4, ring_lane = ring + (uint32_t)(lane >> 3) * 32, col_lane = lds0 + col_b;
    const char *quad = (const char *)(A.recs + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)A.first[stream]) * DR_REC);
    auto ask = [&](uint32_t slot) {
      sp_fill4((const uint32_t *)quad, rec_lane, ring + slot);
      quad += 256;
    };
    int rows = (int)A.Tn;
    fill(rows);
#pragma unroll
    for (int i = 0; i < DR_RING; ++i) ask((uint32_t)i * 256);
    const auto stream_counts = (const __attribute__((address_space(4))) uint4 *)(uintptr_t)A.counts + (int64_t)stream * A.p.stages;
    auto count_at = [&](int at) {
      return mine ? make_uint4(stream_counts[at].x, stream_counts[at].y, stream_counts[at].z, stream_counts[at].w) : make_uint4(0u, 0u, 0u, 0u);
    };
    uint4 cnt = count_at(0);
    asm volatile("s_waitcnt vmcnt(0)" ::"s"(cnt.x), "s"(cnt.y), "s"(cnt.z), "s"(cnt.w) : "memory");
    dr_u32x16_t words;                                     // as in k_decode_rows
    {
      const auto q = (const __attribute__((address_space(3))) u32x4_t *)(uintptr_t)ring_lane;
      const u32x4_t a = q[0], b = q[1];
      words = __builtin_shufflevector(__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7), __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7),
                                      0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
      asm volatile("" ::"v"(words));                       // the slot has been read
      ask(0);
    }
    uint32_t slot = 256, at = 0;
    for (int st = 0; st < A.p.tiles; ++st) {
      if (st > 0) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();                      // nobody reads the last tile any more
        asm volatile("" ::: "memory");
        tile += SP_ROWS * (uint64_t)pitch_b;
        rows -= SP_ROWS;
        fill(rows);
        cnt = count_at(st);                                // (arrives before the tile does)
        asm volatile("s_waitcnt vmcnt(0)" ::"s"(cnt.x), "s"(cnt.y), "s"(cnt.z), "s"(cnt.w) : "memory");
      }
      asm volatile("" ::"v"(words) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      uint32_t n, m0, since;
      at = __builtin_amdgcn_readfirstlane(at);
      slot = __builtin_amdgcn_readfirstlane(slot);
      uint64_t next = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)(uintptr_t)quad >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint64_t)(uintptr_t)quad);
      // (one buffer: no tile comes in meanwhile, and the records' buffer bit is left out)
      DR_STAGE_ASM(0x0FF80u, tile, SP_NO_TILE, 0u, 0u, 0u, 0u);
      quad = (const char *)(uintptr_t)next;
      const uint32_t even = (cnt.x & 0x00FF00FFu) + (cnt.y & 0x00FF00FFu) + (cnt.z & 0x00FF00FFu) + (cnt.w & 0x00FF00FFu);
      const uint32_t odd = ((cnt.x >> 8) & 0x00FF00FFu) + ((cnt.y >> 8) & 0x00FF00FFu) + ((cnt.z >> 8) & 0x00FF00FFu) + ((cnt.w >> 8) & 0x00FF00FFu);
      at += (even + odd) + ((even + odd) >> 16);           // (only its low three bits are looked at)
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may be on its way into LDS when the workgroup ends
  }
  if (!mine) return;

  // lane 8 j + i: of the features of one half, row j, columns 4 i .. 4 i + 3
  const int64_t c = (int64_t)cp * DR_COLS + (lane & 7) * 4;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int64_t f = (int64_t)g * DR_TOK + half * 8 + (lane >> 3);
    const bool on = f < A.F;
    const int64_t at = ((int64_t)slot_dec * A.F) * A.d + c / 8 * A.m_cols + (on ? f : A.F - 1) * A.m_row + c % 8;
    float *const w_at = A.w + ((int64_t)slot_dec * A.F + (on ? f : A.F - 1)) * A.pitch + c;
    f32x4v_t mm = __builtin_nontemporal_load(reinterpret_cast<const f32x4v_t *>(A.m + at));
    f32x4v_t vv = __builtin_nontemporal_load(reinterpret_cast<const f32x4v_t *>(A.v + at));
    f32x4v_t ww = __builtin_nontemporal_load(reinterpret_cast<const f32x4v_t *>(w_at));
    // the eight partial sums of eight rows: a lane gives away half of its rows at each step
    float sum[8][4];
#pragma unroll
    for (int i = 0; i < 32; ++i) sum[i >> 2][i & 3] = half ? hi[i] : lo[i];
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) {
      const bool up = (lane >> 3) & o;
#pragma unroll
      for (int k = 0; k < o; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float keep = up ? sum[k + o][q] : sum[k][q], give = up ? sum[k][q] : sum[k + o][q];
          sum[k][q] = keep + __shfl_xor(give, o * 8);
        }
    }
    f32x4v_t gr{sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
    const float z = fmaf(gr[0], 0.0f, fmaf(gr[1], 0.0f, fmaf(gr[2], 0.0f, gr[3] * 0.0f)));
    // Rows that are not finite once more without the places that fill records up: 0 * inf of such a place gives a NaN.
    for (uint64_t again = ballot64(on && z != z); again != 0;) {
      const int row = __ffsll((unsigned long long)again) - 1 >> 3;
      again &= ~(0xFFull << (8 * row));
      f32x4v_t a{0.f, 0.f, 0.f, 0.f};
      const int32_t *lp = A.list_ptr + (int64_t)s * A.F + (int64_t)g * DR_TOK + half * 8 + row;
      for (int32_t j = lp[0] + (lane >> 3); j < lp[1]; j += DR_REC) {
        const f32x4v_t x = *reinterpret_cast<const f32x4v_t *>(A.g + ((int64_t)t * A.Tn + A.list_tok[j]) * A.d + c);
        const float value = A.val[A.list_src[j]];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = fmaf(value, x[q], a[q]);
      }
#pragma unroll
      for (int o = 8; o < 64; o <<= 1)
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] += __shfl_xor(a[q], o);
      if ((lane >> 3) == row) gr = a;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float m1 = mm[q], v1 = vv[q];
      ww[q] = adam_update(ww[q], gr[q], m1, v1, A.adam);
      mm[q] = m1;
      vv[q] = v1;
    }
    if (on) {
      __builtin_nontemporal_store(mm, reinterpret_cast<f32x4v_t *>(A.m + at));
      __builtin_nontemporal_store(vv, reinterpret_cast<f32x4v_t *>(A.v + at));
      *reinterpret_cast<f32x4v_t *>(w_at) = ww;
    }
  }
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

struct RowLayout {
  RowPlan p;
  int col_parts;
  int64_t n_recs;
  size_t start, counts, offset, total, recs, bytes;
};

static RowLayout row_layout(int64_t Tn, int64_t d, int64_t F, int64_t L, int64_t entries) {
  RowLayout l;
  RowPlan &p = l.p;
  p.tiles = (int)clt_ceil_div(F, SP_ROWS);
  p.groups = (int)clt_ceil_div(Tn, DR_TOK);
  p.stages = (int)(L * p.tiles);
  p.by_layer = 0;
  p.parts = (int)clt_ceil_div(p.groups, DR_WAVES);
  p.groups_per_part = (int)clt_ceil_div(p.groups, p.parts);
  l.col_parts = (int)(d / DR_COLS);
  // every run may leave its last record part empty, but no more runs than entries; every stream its last quad; and a stream reads
  // a ring past its end
  const int64_t runs = (int64_t)p.stages * p.groups * DR_TOK;
  l.n_recs = entries / DR_REC + (runs < entries ? runs : entries) + (DR_RING + 2) * 4;
  size_t at = 0;
  auto take = [&](size_t n) { const size_t here = at; at += align256(n); return here; };
  l.start = take(sizeof(int32_t) * (size_t)L * p.groups * DR_TOK * (p.tiles + 1));
  l.counts = take(sizeof(uint4) * (size_t)p.groups * p.stages);
  l.offset = take(sizeof(uint32_t) * (size_t)p.groups * p.stages);
  l.total = take(sizeof(uint32_t) * (size_t)p.groups);
  l.recs = take((size_t)(l.n_recs + (int64_t)(DR_QUAD - 1) * p.groups) * DR_REC * sizeof(uint2));
  l.bytes = at;
  return l;
}

static RowLayout grad_row_layout(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries) {
  RowLayout l;
  RowPlan &p = l.p;
  p.tiles = (int)clt_ceil_div(T, SP_ROWS);
  p.groups = (int)clt_ceil_div(F, DR_TOK);
  p.stages = p.tiles;
  p.by_layer = 1;
  p.parts = (int)clt_ceil_div(p.groups, GR_WAVES);
  p.groups_per_part = GR_WAVES;
  l.col_parts = (int)(d / DR_COLS);
  const int64_t streams = L * p.groups, runs = streams * p.tiles * DR_TOK;
  l.n_recs = entries / DR_REC + (runs < entries ? runs : entries) + (DR_QUAD - 1) * streams + (DR_RING + 2) * 4;
  size_t at = 0;
  auto take = [&](size_t n) { const size_t here = at; at += align256(n); return here; };
  l.start = take(sizeof(int32_t) * (size_t)streams * DR_TOK * (p.tiles + 1));
  l.counts = take(sizeof(uint4) * (size_t)streams * p.tiles);
  l.offset = take(sizeof(uint32_t) * (size_t)streams * p.tiles);
  l.total = take(sizeof(uint32_t) * (size_t)streams);
  l.recs = take((size_t)l.n_recs * DR_REC * sizeof(uint2));
  l.bytes = at;
  return l;
}
static bool grad_row_shape_ok(const RowLayout &l, int64_t d, int64_t L) {
  return l.p.tiles <= DR_MAX_TILES && l.n_recs <= 0x03FFFFFFll && d * 4 * SP_ROWS <= 0x7FFFFFFFll && l.p.groups <= 0xFFFF &&
         L * l.p.groups * l.p.tiles <= 0x07FFFFFFll && 8 * clt_ceil_div((int64_t)l.p.parts * l.col_parts, 8) * (L * (L + 1) / 2) <= 0x7FFFFFFFll;
}

// LDS for the run starts of every tile; 32-bit offsets of records and of rows within a tile
static bool row_shape_ok(const RowLayout &l, int64_t row_bytes) {
  return l.p.tiles <= DR_MAX_TILES && l.n_recs <= 0x03FFFFFFll && row_bytes * SP_ROWS <= 0x7FFFFFFFll && l.p.groups <= 0xFFFF &&
         (int64_t)l.p.stages * l.p.groups <= 0x07FFFFFFll;
}

}  // namespace

// Priced from what it measured (2496 of the shapes of clt_decode_gather_us; off by 10 % in the mean): a stage of the tiles takes 1.2 us plus
// 5 ns per record, but no less than 64 KB take to come into LDS, 2.0 us from HBM and 1.3 where the targets share a decoder; workgroups of
// unequal length end a quarter of the longest behind the mean, and the longest one bounds a launch of few.  us, tiles / gather: L = 12, d =
// 768, F = 6144: 1469 / 2618 with 200 per token at T = 1024, 949 / 1198 with 60, 805 / 717 with 20; 647 / 1112 with 200 at 256; L =
// 6, d = 1024, F = 16384: 2519 / 2796 at 3000 x 200, 2169 / 1704 at 3000 x 100; L = 16, d = 256, F = 2048, 1024 x 30: 234 / 565.
double clt_decode_rows_us(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying, int dtype) {
  const double no = 1e30;
  if (dtype != CLT_F32 || (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE)) return no;
  if (T <= 0 || d <= 0 || d % DR_COLS != 0 || F <= 0 || L <= 0 || L > 64 || targets <= 0 || targets > L || entries <= 0) return no;
  const RowLayout l = row_layout(T, d, F, L, entries);
  if (!row_shape_ok(l, clt_pitch(d, 4) * 4)) return no;
  const double pairs = 0.5 * targets * (2 * L - targets + 1), run = (double)entries / ((double)l.p.stages * T);
  const double recs = l.p.groups_per_part * DR_TOK * (run < run / DR_REC + 0.29 ? run : run / DR_REC + 0.29);
  const double stage = 1.16 + recs * 0.005, fill = tying == CLT_TYING_NONE ? 1.97 : 1.3;
  const double stages = pairs * l.p.tiles * l.col_parts * l.p.parts / 256, longest = (double)L * l.p.tiles;
  const double last = stages + 0.28 * longest > longest ? stages + 0.28 * longest : longest;
  return last * (stage > fill ? stage : fill) + 27 + entries * 1.5e-5;
}

extern "C" int clt_decode_rows_wanted(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying,
                                      int dtype) {
  const double us = clt_decode_rows_us(T, d, F, L, targets, entries, tying, dtype);
  return us < 1e30 && us < 0.95 * clt_decode_gather_us(T, d, F, L, targets, entries, tying, dtype);
}

extern "C" size_t clt_decode_rows_workspace_bytes(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries) {
  if (T <= 0 || d < DR_COLS || F <= 0 || L <= 0 || entries < 0) return 0;
  return row_layout(T, d, F, L, entries).bytes;
}

extern "C" int clt_decode_rows(const int32_t *row_ptr, const int32_t *col, const float *val, const float *w_packed,
                               const float *bias_sum, const float *skip_add, float *out, int64_t T, int64_t d, int64_t F, int64_t L,
                               int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int64_t entries, void *workspace,
                               size_t workspace_bytes, void *stream) {
  if (T < 0 || d <= 0 || F <= 0 || L <= 0 || L > 64 || d % DR_COLS != 0 || entries < 0) return CLT_ERR_ARG;
  if (t_begin < 0 || t_end > L || t_begin > t_end) return CLT_ERR_ARG;
  if (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE) return CLT_ERR_ARG;
  if (T == 0 || t_begin == t_end) return CLT_OK;
  if (!row_ptr || !col || !val || !w_packed || !out || !workspace) return CLT_ERR_ARG;
  if (!clt_aligned16(w_packed) || !clt_aligned16(out) || !clt_aligned16(workspace) || (bias_sum && !clt_aligned16(bias_sum)) ||
      (skip_add && !clt_aligned16(skip_add)))
    return CLT_ERR_ALIGN;
  const int64_t pitch = clt_pitch(d, 4);
  const RowLayout l = row_layout(T, d, F, L, entries);
  if (!row_shape_ok(l, pitch * 4)) return CLT_ERR_RANGE;
  if (workspace_bytes < l.bytes) return CLT_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  char *ws = (char *)workspace;
  RunArgs ra;
  ra.row_ptr = row_ptr; ra.col = col; ra.src = nullptr; ra.val = val; ra.Tn = T; ra.L = L; ra.max_entries = entries; ra.layer_mask = src_mask; ra.p = l.p;
  ra.start = (int32_t *)(ws + l.start); ra.counts = (uint4 *)(ws + l.counts); ra.offset = (uint32_t *)(ws + l.offset);
  ra.total = (uint32_t *)(ws + l.total); ra.recs = (uint2 *)(ws + l.recs);
  RowArgs a;
  a.p = l.p; a.counts = ra.counts; a.total = ra.total; a.recs = ra.recs;
  a.wp = w_packed; a.bias_sum = bias_sum; a.skip_add = skip_add; a.out = out;
  a.row_ptr = row_ptr; a.col = col; a.val = val;
  a.Tn = T; a.d = d; a.F = F; a.L = L; a.pitch = pitch; a.max_entries = entries; a.src_mask = src_mask;
  a.tying = tying; a.t_begin = (int)t_begin; a.t_end = (int)t_end; a.col_parts = l.col_parts;
  const int64_t pairs = clt_ceil_div((t_end - t_begin) * l.col_parts, 8) * 8;
  if (pairs * l.p.parts > 0x7FFFFFFFll) return CLT_ERR_RANGE;
  if (hipFuncSetAttribute((const void *)k_decode_rows, hipFuncAttributeMaxDynamicSharedMemorySize, DR_LDS) != hipSuccess)
    return CLT_ERR_LAUNCH;
  const size_t run_lds = sizeof(int32_t) * (size_t)DR_TOK * (l.p.tiles + 1);
  const dim3 grid((unsigned)l.p.groups, (unsigned)L);
  const size_t fill_bytes = run_lds + sizeof(uint32_t) * (size_t)DR_TOK * l.p.tiles;
  if (hipFuncSetAttribute((const void *)k_row_fill, hipFuncAttributeMaxDynamicSharedMemorySize, (int)fill_bytes) != hipSuccess)
    return CLT_ERR_LAUNCH;
  k_row_runs<<<grid, DR_THREADS, run_lds, s>>>(ra);
  k_row_streams<<<(unsigned)l.p.groups, 64, 0, s>>>(ra);
  k_row_fill<<<grid, DR_THREADS, fill_bytes, s>>>(ra);
  k_decode_rows<<<(unsigned)(pairs * l.p.parts), DR_WAVES * 64, DR_LDS, s>>>(a);
  return clt_check_launch();
}

extern "C" int clt_grad_rows_supported(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries, int dtype) {
  if (dtype != CLT_F32 || T <= 0 || d <= 0 || d % DR_COLS != 0 || F <= 0 || L <= 0 || L > 64 || entries <= 0) return 0;
  return grad_row_shape_ok(grad_row_layout(T, d, F, L, entries), d, L);
}

// Measured at 46 shapes (L 2 - 16, d 256 - 2048, F 256 - 32768, T 32 - 8192) against the other in-place steps of float32 decoders, by the
// entries of a list.  A tile takes some 4 us whatever it holds, so few entries do not pay for many tiles: from 9 per tile on
// (8 for up to two tiles) this is the fastest or second to rows by microseconds.  Lists of fewer than 8 go row by row: nothing is
// regrouped, and few rows are gathered.  us, here / 32-byte tiles / rows: L = 12, d = 768, F = 6144, T = 1024: 2602 / 3926 / 4036 with 33
// entries, 2285 / 2682 / 2553 with 13, 2216 / 2357 / 1891 with 5; T = 4096: 7853 / 13002 / 21267 with 133, 7209 / 3130 / 4359 with 20; L
// = 8, d = 1024, F = 8192, T = 4096: 6042 / 7208 / 13117 with 90, 5877 / 4489 / 7872 with 50; L = 6, d = 1024, F = 16384, T = 1500: 3199 / 2217 /
// 1657 with 3; L = 6, d = 512, F = 8192, T = 3000: 1104 / 605 / 549 with 7.  Launches that do not fill the chip once are left as they were.
extern "C" int clt_grad_rows_wanted(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries, int dtype) {
  if (!clt_grad_rows_supported(T, d, F, L, entries, dtype)) return 0;
  const RowLayout l = grad_row_layout(T, d, F, L, entries);
  if ((int64_t)l.p.parts * l.col_parts * (L * (L + 1) / 2) < 512) return 0;
  const double per_list = (double)entries / ((double)L * F);
  if (per_list < 8) return 2;
  return l.p.tiles <= 2 || per_list >= 9.0 * l.p.tiles;
}

extern "C" size_t clt_grad_rows_workspace_bytes(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries) {
  if (T <= 0 || d < DR_COLS || F <= 0 || L <= 0 || entries <= 0) return 0;
  return grad_row_layout(T, d, F, L, entries).bytes;
}

extern "C" int clt_decoder_grad_adam_rows(const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const float *val,
                                          const float *g, float *w_packed, float *m, float *v, int moments_by_tile, int64_t T, int64_t d,
                                          int64_t F, int64_t L, int64_t entries, double lr, double beta1, double beta2, double eps,
                                          int64_t step, void *workspace, size_t workspace_bytes, void *stream) {
  if (!clt_grad_rows_supported(T, d, F, L, entries, CLT_F32)) return CLT_ERR_ARG;
  if (step < 1 || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1)) return CLT_ERR_ARG;
  if (!list_ptr || !list_tok || !list_src || !val || !g || !w_packed || !m || !v || !workspace) return CLT_ERR_ARG;
  if (!clt_aligned16(g) || !clt_aligned16(w_packed) || !clt_aligned16(m) || !clt_aligned16(v) || !clt_aligned16(workspace)) return CLT_ERR_ALIGN;
  const RowLayout l = grad_row_layout(T, d, F, L, entries);
  if (workspace_bytes < l.bytes) return CLT_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  char *ws = (char *)workspace;
  RunArgs ra;
  ra.row_ptr = list_ptr; ra.col = list_tok; ra.src = list_src; ra.val = val; ra.Tn = F; ra.L = L; ra.max_entries = entries; ra.layer_mask = ~0ull; ra.p = l.p;
  ra.start = (int32_t *)(ws + l.start); ra.counts = (uint4 *)(ws + l.counts); ra.offset = (uint32_t *)(ws + l.offset);
  ra.total = (uint32_t *)(ws + l.total); ra.recs = (uint2 *)(ws + l.recs);
  GradRowArgs a;
  a.p = l.p; a.counts = ra.counts; a.first = ra.total; a.recs = ra.recs;
  a.g = g; a.w = w_packed; a.m = m; a.v = v;
  a.list_ptr = list_ptr; a.list_tok = list_tok; a.list_src = list_src; a.val = val;
  a.Tn = T; a.d = d; a.F = F; a.L = L; a.pitch = clt_pitch(d, 4); a.max_entries = entries;
  a.m_row = moments_by_tile ? 8 : d;
  a.m_cols = moments_by_tile ? F * 8 : 8;
  a.col_parts = l.col_parts;
  a.items = (int)clt_ceil_div((int64_t)l.p.parts * l.col_parts, 8);
  a.adam = adam_coef(lr, beta1, beta2, eps, step);
  const int streams = (int)L * l.p.groups;
  const size_t run_lds = sizeof(int32_t) * (size_t)DR_TOK * (l.p.tiles + 1), fill_bytes = run_lds + sizeof(uint32_t) * (size_t)DR_TOK * l.p.tiles;
  if (hipFuncSetAttribute((const void *)k_grad_rows, hipFuncAttributeMaxDynamicSharedMemorySize, GR_LDS) != hipSuccess ||
      hipFuncSetAttribute((const void *)k_row_fill, hipFuncAttributeMaxDynamicSharedMemorySize, (int)fill_bytes) != hipSuccess)
    return CLT_ERR_LAUNCH;
  const dim3 grid((unsigned)l.p.groups, (unsigned)L);
  k_row_runs<<<grid, DR_THREADS, run_lds, s>>>(ra);
  k_row_streams<<<(unsigned)streams, 64, 0, s>>>(ra);
  k_row_firsts<<<1, DR_FIRSTS, 0, s>>>(ra.total, streams);
  k_row_fill<<<grid, DR_THREADS, fill_bytes, s>>>(ra);
  k_grad_rows<<<(unsigned)(8 * a.items * (L * (L + 1) / 2)), GR_WAVES * 64, GR_LDS, s>>>(a);
  return clt_check_launch();
}
