// Survivor lists regrouped for the matrix cores, and the inner step of the kernels that multiply them.
//
// A sparse product out[row] += sum over entries (row, r, v) of v * W[r][:] is cut into tiles: SP_ROWS consecutive rows
// r of W times SP_COLS columns sit in LDS, and the entries that fall into a tile are grouped by 16 consecutive output
// rows.  32 entries of a group form one batch: a 32 x 16 operand with ONE non-zero per entry (its value in the column
// of its output row) times the 64 x 32 operand made of the entries' W rows, i.e. four 16x16x32 matrix instructions.
// The gathered operand comes out of LDS through the transposing read, which takes an address per lane.
//
// Why: a gather through the vector memory path is bound by the L1's outstanding lines (15 TB/s at best on this part);
// LDS hands out 32-byte pieces at 60 TB/s if they are chosen at random and at 124 if no two of a half wavefront's meet in a bank
// (2.19 and 1.06 ns per 512-byte transposing read and CU; profiles/lds_read_probe.txt).  Fifteen sixteenths of the matrix instruction's products are with zeros,
// which still leaves as many useful ones per cycle as the vector unit's dot products deliver, without their
// unpacking; and lists of unequal length cost nothing, because a batch is filled from any of 16 output rows.
#pragma once
#include <type_traits>
#include "clt_common.h"

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4v_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

constexpr int SP_COLS = 64;          // columns of a tile: one 128-byte line of 16-bit elements
constexpr int SP_ROWS = 512;         // W rows of a tile: 64 KB, and two of them leave 32 KB of the CU's LDS for records
constexpr int SP_TILE_BYTES = SP_ROWS * 128;
constexpr int SP_GROUP = 16;         // output rows of a group
constexpr int SP_BATCH = 32;         // entries of a batch

// A batch's record is one 32-bit word per lane.  Lane 16 q + 4 x + y of the wavefront holds, for entries 8 q .. 8 q + 7:
//   y = 0   values of entries 8 q + 2 x, 8 q + 2 x + 1
//   y = 1   their output rows as one-hot 16-bit masks
//   y = 3   where their tile rows begin in the tile: entry 8 q + x low, entry 8 q + 4 + x high
// - every lane finds what it needs in its own row of 16 lanes, one DPP operand away, so that a record costs one dword of
// LDS traffic per lane beside the eight transposing reads (broadcasting it with two 16-byte reads instead: five vector
// instructions fewer, but a quarter more LDS time per batch).
// The records of four consecutive batches of a stream lie together, a lane's four words next to each other: they come in with
// one load and are read with another.  Streams begin at whole quads.
constexpr int SP_REC_WORDS = 64;
constexpr int SP_QUAD = 4;                           // batches of a quad
constexpr int SP_QUAD_BYTES = SP_QUAD * SP_REC_WORDS * 4;
constexpr int SP_RING_BYTES = 2 * SP_QUAD_BYTES;     // quads that a wavefront keeps in LDS or on their way
// Batches past the end of the last stream that are asked for: three quads are under way or read when the first batch is taken up, and one
// more is asked for whenever a quad is through.
constexpr int SP_PAST_END = 3 * SP_QUAD;
// where word `w` of batch `b` (counted over all streams) lies
__device__ __forceinline__ uint64_t sp_rec_word(uint64_t b, uint32_t w) {
  return (b / SP_QUAD) * (SP_QUAD * SP_REC_WORDS) + w * SP_QUAD + b % SP_QUAD;
}

// A tile lies in LDS as two halves of 32 columns, 64 bytes per row; the two 32-byte pieces of a row are exchanged in
// every other group of four rows, so that one piece of eight consecutive rows covers all banks.  Column piece n of a row
// is then at place ^ 32 (n & 1), plus half a tile for n >= 2: one exclusive-or for two reads, the rest in their offsets.
constexpr int SP_HALF_BYTES = SP_TILE_BYTES / 2;
__host__ __device__ __forceinline__ uint32_t sp_swap(uint32_t r) { return (r >> 2) & 1u; }
__device__ __forceinline__ uint32_t sp_place(uint32_t r) { return (r << 6) | (sp_swap(r) << 5); }

// what the kernels over tiles share: a decoder's place in the slab, a stream's first record, loads into LDS
__device__ __forceinline__ int64_t sp_slot(int tying, int64_t s, int64_t t, int64_t L) {
  return tying == CLT_TYING_PER_SOURCE ? s : s * L - (s * (s - 1)) / 2 + (t - s);
}

// first batch (record) of a stream: those of the streams before it (all lanes of a wavefront take part)
__device__ __forceinline__ uint32_t stream_first(const uint32_t *total, int stream, int lane) {
  uint32_t n = 0;
  for (int i = lane; i < stream; i += 64) n += total[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
  return n;
}

// Direct-to-LDS loads, 16 or 4 bytes per lane (lane i lands at lds_at + 16 i / 4 i).  As asm statements, so that the
// compiler does not wait for them in front of every LDS read; whoever reads the data waits by hand.
__device__ __forceinline__ void sp_fill16(const char *base, uint32_t off, uint32_t lds_at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds_at) : "memory");
}
__device__ __forceinline__ void sp_fill4(const uint32_t *base, uint32_t off, uint32_t lds_at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "{m0}"(lds_at) : "memory");
}

// ---- the batches of one stage -------------------------------------------------------------------------
// What a wavefront does between two barriers: the batches of its four groups that fall into the tile in LDS.  Per batch it turns
// the record's word into addresses (3 vector instructions), sets eight transposing reads going (2), builds the operand of
// values (16) and multiplies (4 matrix instructions).  Two batches are in the making at any time: the reads of the next one are
// asked for before this one is multiplied, so that a wavefront waits for LDS only where a whole batch's time was not enough.
// The last batch of a stage has no successor whose tile is there, and sets no reads going.
//
// One copy of the code for each group and place of a batch in two quads (no selection of registers, jumps only from group to
// group), and the books of the records once per quad: a batch takes 26 vector instructions, 8 reads and some 7 scalar ones, where
// one copy per group with a record at a time takes 27, 9 and 13 (k_decode_tiles at 4096 tokens, L = 12, d = 768, F = 24576: 3.10 ->
// 2.82 ms; k_grad_tiles 7.41 -> 7.16).  Two batches in the making alone, one record at a time: 3.29 ms.
//
// Written in assembly as a whole, because over these loops the compiler keeps neither the 64 sums and the two operands in place
// (it copies or spills them) nor the waits apart.  Registers: v0 - v63 the sums (group g, columns 16 n ..: v[16 g + 4 n ..]),
// v64 - v79 and v80 - v95 the two 64 x 32 operands, v96 - v99 and v100 - v103 their values, v112 - v119 the words of two quads,
// s[40:41] the next quad to ask for.  Nothing is on its way into a register when the block ends.
//
// Lane = 16 q + i supplies entries 8 q .. 8 q + 7 of output row i; of the sums it holds columns 4 q .. 4 q + 3 of output row i.
typedef float f32x32v_t __attribute__((ext_vector_type(32)));
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));
struct SpSums {
  f32x32v_t lo, hi;                        // groups 0, 1 and 2, 3
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 32; ++i) { lo[i] = 0.f; hi[i] = 0.f; }
  }
  __device__ __forceinline__ void get(int g, f32x4v_t (&out)[4]) const {
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i >> 2][i & 3] = g < 2 ? lo[(g & 1) * 16 + i] : hi[(g & 1) * 16 + i];
  }
};

// the places in LDS of the rows that the word W refers to, to v104 and v105
#define SP_ADDRESS(W)                                                                          \
  "v_mov_b32_dpp v104, " W " quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"               \
  "v_add_u32_sdwa v105, v104, %[col] dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1 src1_sel:DWORD\n\t" \
  "v_add_u32_sdwa v104, v104, %[col] dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:DWORD\n\t"
#define SP_READ(A, B, C, D, E, F, G, H)                                                        \
  "v_xor_b32 v106, 32, v104\n\t"                                                               \
  "v_xor_b32 v107, 32, v105\n\t"                                                               \
  "ds_read_b64_tr_b16 v[" A "], v104\n\t"                                                      \
  "ds_read_b64_tr_b16 v[" B "], v105\n\t"                                                      \
  "ds_read_b64_tr_b16 v[" C "], v106\n\t"                                                      \
  "ds_read_b64_tr_b16 v[" D "], v107\n\t"                                                      \
  "ds_read_b64_tr_b16 v[" E "], v104 offset:32768\n\t"                                         \
  "ds_read_b64_tr_b16 v[" F "], v105 offset:32768\n\t"                                         \
  "ds_read_b64_tr_b16 v[" G "], v106 offset:32768\n\t"                                         \
  "ds_read_b64_tr_b16 v[" H "], v107 offset:32768\n\t"
#define SP_READ_0 SP_READ("64:65", "66:67", "68:69", "70:71", "72:73", "74:75", "76:77", "78:79")
#define SP_READ_1 SP_READ("80:81", "82:83", "84:85", "86:87", "88:89", "90:91", "92:93", "94:95")
static_assert(SP_HALF_BYTES == 32768, "written out above");
// Values of two of the lane's eight entries where they belong to its output row, zero elsewhere: one-hot & row_bit (bit i of
// both halves) is non-zero there, and min(.., 1) is a factor.
#define SP_PICK(P, T, W, HOT, VAL)                                                             \
  "v_and_b32_dpp " P ", " W ", %[row_bit] row_newbcast:" HOT " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mov_b32_dpp " T ", " W " row_newbcast:" VAL " row_mask:0xf bank_mask:0xf\n\t"             \
  "v_pk_min_u16 " P ", " P ", %[ones]\n\t"                                                     \
  "v_pk_mul_lo_u16 " P ", " P ", " T "\n\t"
#define SP_PICK_0A(W) SP_PICK("v96", "v108", W, "1", "0")
#define SP_PICK_0B(W) SP_PICK("v97", "v109", W, "5", "4")
#define SP_PICK_0C(W) SP_PICK("v98", "v108", W, "9", "8")
#define SP_PICK_0D(W) SP_PICK("v99", "v109", W, "13", "12")
#define SP_PICK_1A(W) SP_PICK("v100", "v108", W, "1", "0")
#define SP_PICK_1B(W) SP_PICK("v101", "v109", W, "5", "4")
#define SP_PICK_1C(W) SP_PICK("v102", "v108", W, "9", "8")
#define SP_PICK_1D(W) SP_PICK("v103", "v109", W, "13", "12")
#define SP_MUL(M, C, A, B) M " v[" C "], v[" A "], v[" B "], v[" C "]\n\t"
#define SP_MUL_0A(M, C) SP_MUL(M, C, "64:67", "96:99")
#define SP_MUL_0B(M, C) SP_MUL(M, C, "68:71", "96:99")
#define SP_MUL_0C(M, C) SP_MUL(M, C, "72:75", "96:99")
#define SP_MUL_0D(M, C) SP_MUL(M, C, "76:79", "96:99")
#define SP_MUL_1A(M, C) SP_MUL(M, C, "80:83", "100:103")
#define SP_MUL_1B(M, C) SP_MUL(M, C, "84:87", "100:103")
#define SP_MUL_1C(M, C) SP_MUL(M, C, "88:91", "100:103")
#define SP_MUL_1D(M, C) SP_MUL(M, C, "92:95", "100:103")

// The records.  At places 2 and 6 of a stream's batches the next quad is read from its slot of the ring (the other quad was asked
// for since, and perhaps the four loads of a tile if fewer than two quads were asked for after those); a place later it has
// arrived (a batch's eight reads were asked for behind it), and its slot goes to the quad after the one in the other slot.
#define SP_RING_READ(G, P, TO, AT)                                                             \
  "s_cmp_lt_i32 %[since], 2\n\t"                                                               \
  "s_cbranch_scc1 .Lsp_v" G P "_%=\n\t"                                                        \
  "s_waitcnt vmcnt(1)\n"                                                                       \
  ".Lsp_v" G P "_%=:\n\t"                                                                      \
  "s_waitcnt vmcnt(5)\n\t"                                                                     \
  "ds_read_b128 v[" TO "], %[ring_lane] offset:" AT "\n\t"
#define SP_RING_ASK(SET_M0)                                                                    \
  "s_waitcnt lgkmcnt(8)\n\t" SET_M0                                                            \
  "s_add_i32 %[since], %[since], 1\n\t"                                                        \
  "global_load_lds_dwordx4 %[ring_lane], s[40:41]\n\t"                                         \
  "s_add_u32 s40, s40, 0x400\n\t"                                                              \
  "s_addc_u32 s41, s41, 0\n\t"
#define SP_BOOKS_0(G)
#define SP_BOOKS_1(G)
#define SP_BOOKS_2(G) SP_RING_READ(G, "2", "116:119", "1024")
#define SP_BOOKS_3(G) SP_RING_ASK("s_add_i32 m0, %[ring], 0x400\n\t")
#define SP_BOOKS_4(G)
#define SP_BOOKS_5(G)
#define SP_BOOKS_6(G) SP_RING_READ(G, "6", "112:115", "0")
#define SP_BOOKS_7(G) SP_RING_ASK("s_mov_b32 m0, %[ring]\n\t")
static_assert(SP_QUAD_BYTES == 1024, "written out above");
// reads under way behind those of the batch that is multiplied: its successor's eight and a quad's; without a successor
#define SP_BEHIND_0 "8"
#define SP_BEHIND_1 "8"
#define SP_BEHIND_2 "9"
#define SP_BEHIND_3 "8"
#define SP_BEHIND_4 "8"
#define SP_BEHIND_5 "8"
#define SP_BEHIND_6 "9"
#define SP_BEHIND_7 "8"
#define SP_ALONE_0 "0"
#define SP_ALONE_1 "0"
#define SP_ALONE_2 "1"
#define SP_ALONE_3 "0"
#define SP_ALONE_4 "0"
#define SP_ALONE_5 "0"
#define SP_ALONE_6 "1"
#define SP_ALONE_7 "0"

// The batch at place P of group G (sums C0 .. C3), and its successor at place N with the word W: it is multiplied from set S while
// the successor is prepared in set R.  `n`: batches of the group still to come behind it.
#define SP_BATCH_CODE(M, G, P, N, S, R, W, C0, C1, C2, C3)                                     \
  ".Lsp_b" G #P "_%=:\n\t"                                                                     \
  SP_BOOKS_##P(G) SP_ADDRESS(W) SP_READ_##R                                                    \
  "s_waitcnt lgkmcnt(" SP_BEHIND_##P ")\n\t"                                                   \
  SP_MUL_##S##A(M, C0) SP_PICK_##R##A(W)                                                       \
  SP_MUL_##S##B(M, C1) SP_PICK_##R##B(W)                                                       \
  SP_MUL_##S##C(M, C2) SP_PICK_##R##C(W)                                                       \
  SP_MUL_##S##D(M, C3) SP_PICK_##R##D(W)                                                       \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                \
  "s_cbranch_scc1 .Lsp_x" G #N "_%=\n"
// the stage's last batch, of this group and at this place
#define SP_LAST_CODE(M, G, P, S, C0, C1, C2, C3)                                               \
  ".Lsp_l" G #P "_%=:\n\t"                                                                     \
  SP_BOOKS_##P("l" G)                                                                          \
  "s_waitcnt lgkmcnt(" SP_ALONE_##P ")\n\t"                                                    \
  SP_MUL_##S##A(M, C0) SP_MUL_##S##B(M, C1) SP_MUL_##S##C(M, C2) SP_MUL_##S##D(M, C3)          \
  "s_branch .Lsp_end_%=\n"
// behind group G, at place P: group NEXT, whose number of batches is taken out of the stage's counts (borrowing if there is none)
#define SP_SWITCH_CODE(G, NEXT, COUNT, P)                                                      \
  ".Lsp_x" G #P "_%=:\n\t"                                                                     \
  "s_bfe_u32 %[n], " COUNT "\n\t"                                                              \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                \
  "s_cbranch_scc0 .Lsp_b" NEXT #P "_%=\n\t"                                                    \
  "s_branch .Lsp_x" NEXT #P "_%=\n"
#define SP_GROUP_CODE(M, G, C0, C1, C2, C3)                                                    \
  SP_BATCH_CODE(M, G, 0, 1, 0, 1, "v113", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 1, 2, 1, 0, "v114", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 2, 3, 0, 1, "v115", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 3, 4, 1, 0, "v116", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 4, 5, 0, 1, "v117", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 5, 6, 1, 0, "v118", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 6, 7, 0, 1, "v119", C0, C1, C2, C3)                                      \
  SP_BATCH_CODE(M, G, 7, 0, 1, 0, "v112", C0, C1, C2, C3)                                      \
  "s_branch .Lsp_b" G "0_%=\n"                                                                 \
  SP_LAST_CODE(M, G, 0, 0, C0, C1, C2, C3) SP_LAST_CODE(M, G, 1, 1, C0, C1, C2, C3)            \
  SP_LAST_CODE(M, G, 2, 0, C0, C1, C2, C3) SP_LAST_CODE(M, G, 3, 1, C0, C1, C2, C3)            \
  SP_LAST_CODE(M, G, 4, 0, C0, C1, C2, C3) SP_LAST_CODE(M, G, 5, 1, C0, C1, C2, C3)            \
  SP_LAST_CODE(M, G, 6, 0, C0, C1, C2, C3) SP_LAST_CODE(M, G, 7, 1, C0, C1, C2, C3)
#define SP_SWITCH_CODES(G, NEXT, COUNT)                                                        \
  SP_SWITCH_CODE(G, NEXT, COUNT, 0) SP_SWITCH_CODE(G, NEXT, COUNT, 1)                          \
  SP_SWITCH_CODE(G, NEXT, COUNT, 2) SP_SWITCH_CODE(G, NEXT, COUNT, 3)                          \
  SP_SWITCH_CODE(G, NEXT, COUNT, 4) SP_SWITCH_CODE(G, NEXT, COUNT, 5)                          \
  SP_SWITCH_CODE(G, NEXT, COUNT, 6) SP_SWITCH_CODE(G, NEXT, COUNT, 7)
// behind the last group: the stage's last batch is still to come, of group SP_LAST
#define SP_FINISH_CODE(P)                                                                      \
  ".Lsp_x3" #P "_%=:\n\t"                                                                      \
  "s_bfe_u32 %[n], %[cy], 0x2000a\n\t"                                                         \
  "s_cmp_eq_u32 %[n], 3\n\ts_cbranch_scc1 .Lsp_l3" #P "_%=\n\t"                                \
  "s_cmp_eq_u32 %[n], 2\n\ts_cbranch_scc1 .Lsp_l2" #P "_%=\n\t"                                \
  "s_cmp_eq_u32 %[n], 1\n\ts_cbranch_scc1 .Lsp_l1" #P "_%=\n\t"                                \
  "s_branch .Lsp_l0" #P "_%=\n"
// four loads of the tile after this one, if there is one
#define SP_FILL                                                                                \
  "s_mov_b32 m0, %[to]\n\t"                                                                    \
  "s_mov_b32 %[since], 0\n\t"                                                                  \
  "global_load_lds_dwordx4 %[off0], %[from0]\n\t"                                              \
  "s_add_i32 m0, %[to], 0x8000\n\t"                                                            \
  "s_nop 0\n\t"                                                                                \
  "global_load_lds_dwordx4 %[off0], %[from1]\n\t"                                              \
  "s_add_i32 m0, %[to], 0x400\n\t"                                                             \
  "s_nop 0\n\t"                                                                                \
  "global_load_lds_dwordx4 %[off1], %[from0]\n\t"                                              \
  "s_add_i32 m0, %[to], 0x8400\n\t"                                                            \
  "s_nop 0\n\t"                                                                                \
  "global_load_lds_dwordx4 %[off1], %[from1]\n"
#define SP_FILL_IF(L)                                                                          \
  "s_mov_b32 %[since], 2\n\t"                                                                  \
  "s_cmp_eq_i32 %[to], -1\n\t"                                                                 \
  "s_cbranch_scc1 .Lsp_f" L "_%=\n\t"                                                          \
  SP_FILL ".Lsp_f" L "_%=:\n\t"
#define SP_FILL_NONE(L) "s_mov_b32 %[since], 2\n\t"
// the stage's first batch, at place P and with the word W: its tile is there
#define SP_ENTER_CODE(FILL, P, S, W)                                                              \
  ".Lsp_e" #P "_%=:\n\t"                                                                       \
  SP_ADDRESS(W) SP_READ_##S FILL(#P)                                                     \
  SP_PICK_##S##A(W) SP_PICK_##S##B(W) SP_PICK_##S##C(W) SP_PICK_##S##D(W)                      \
  "s_bfe_u32 %[n], %[cx], 0xa0000\n\t"                                                         \
  "s_sub_u32 %[n], %[n], 1\n\t"                                                                \
  "s_cbranch_scc0 .Lsp_b0" #P "_%=\n\t"                                                        \
  "s_branch .Lsp_x0" #P "_%=\n"
#define SP_STAGE(M, FILL)                                                                      \
  "s_lshr_b32 %[n], %[cy], 16\n\t"                                                             \
  "s_cmp_eq_u32 %[n], 0\n\ts_cbranch_scc1 .Lsp_none_%=\n\t"                                    \
  "s_bitcmp1_b32 %[at], 2\n\ts_cbranch_scc1 .Lsp_eb_%=\n\t"                                    \
  "s_bitcmp1_b32 %[at], 1\n\ts_cbranch_scc1 .Lsp_ea_%=\n\t"                                    \
  "s_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Lsp_e1_%=\n"                                      \
  SP_ENTER_CODE(FILL, 0, 0, "v112") SP_ENTER_CODE(FILL, 1, 1, "v113")                                      \
  ".Lsp_ea_%=:\n\ts_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Lsp_e3_%=\n"                       \
  SP_ENTER_CODE(FILL, 2, 0, "v114") SP_ENTER_CODE(FILL, 3, 1, "v115")                                      \
  ".Lsp_eb_%=:\n\ts_bitcmp1_b32 %[at], 1\n\ts_cbranch_scc1 .Lsp_ec_%=\n\t"                     \
  "s_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Lsp_e5_%=\n"                                      \
  SP_ENTER_CODE(FILL, 4, 0, "v116") SP_ENTER_CODE(FILL, 5, 1, "v117")                                      \
  ".Lsp_ec_%=:\n\ts_bitcmp1_b32 %[at], 0\n\ts_cbranch_scc1 .Lsp_e7_%=\n"                       \
  SP_ENTER_CODE(FILL, 6, 0, "v118") SP_ENTER_CODE(FILL, 7, 1, "v119")                                      \
  SP_GROUP_CODE(M, "0", "0:3", "4:7", "8:11", "12:15") SP_SWITCH_CODES("0", "1", "%[cx], 0xa000a")     \
  SP_GROUP_CODE(M, "1", "16:19", "20:23", "24:27", "28:31") SP_SWITCH_CODES("1", "2", "%[cx], 0xa0014") \
  SP_GROUP_CODE(M, "2", "32:35", "36:39", "40:43", "44:47") SP_SWITCH_CODES("2", "3", "%[cy], 0xa0000") \
  SP_GROUP_CODE(M, "3", "48:51", "52:55", "56:59", "60:63")                                    \
  SP_FINISH_CODE(0) SP_FINISH_CODE(1) SP_FINISH_CODE(2) SP_FINISH_CODE(3)                      \
  SP_FINISH_CODE(4) SP_FINISH_CODE(5) SP_FINISH_CODE(6) SP_FINISH_CODE(7)                      \
  ".Lsp_none_%=:\n\t" FILL("n")                                                          \
  ".Lsp_end_%=:\n\t"                                                                           \
  "s_lshr_b32 %[n], %[cy], 16\n\t"                                                             \
  "s_add_u32 %[at], %[at], %[n]\n\t"                                                           \
  "s_cmp_ge_i32 %[since], 2\n\t"   /* the tile's lines, not the quads asked for behind them */ \
  "s_cbranch_scc1 .Lsp_two_%=\n\t"                                                             \
  "s_waitcnt vmcnt(0)\n"                                                                       \
  ".Lsp_two_%=:\n\t"                                                                           \
  "s_waitcnt vmcnt(2) lgkmcnt(0)\n\t"                                                          \
  "s_nop 7\n\ts_nop 7"             /* the last product is there for whoever reads the sums */

// A stage's counts, as k_rec_streams leaves them for each stream: ten bits for each group, without the stage's last batch; the
// group that one belongs to; and all together.
__device__ __forceinline__ uint2 sp_stage_counts(uint32_t n0, uint32_t n1, uint32_t n2, uint32_t n3) {
  const uint32_t all = n0 + n1 + n2 + n3, last = n3 ? 3u : n2 ? 2u : n1 ? 1u : 0u;
  if (all) (last == 3 ? n3 : last == 2 ? n2 : last == 1 ? n1 : n0) -= 1;
  return make_uint2(n0 | (n1 << 10) | (n2 << 20), n3 | (last << 10) | (all << 16));
}
static_assert(SP_GROUP * SP_ROWS / SP_BATCH < 1024, "ten bits");

// A wavefront's four loads of a tile: where the tile begins, the lane's places there, the share's place in LDS (SP_NO_TILE: there
// is no tile).
constexpr uint32_t SP_NO_TILE = ~0u;
struct SpFill { const char *from; uint32_t off0, off1, to; };
struct SpNoFill {};

// A wavefront's place in its stream of batches.
struct SpStream {
  const char *next;                        // the next quad to ask for, less `ring`
  uint32_t ring, ring_lane;                // the ring in LDS; the lane's words of its first quad
  uint32_t at;                             // the batch that comes next
  u32x8_t words;                           // of the quads at hand
  uint32_t col, row_bit;                   // where the tile at hand begins in LDS plus 8 * (lane % 4); bit (lane % 16) of both halves

  // Quad `slot` of the ring, on its way in.
  __device__ __forceinline__ void ask(uint32_t slot) {
    sp_fill16(next, ring_lane, ring + slot * SP_QUAD_BYTES);
    next += SP_QUAD_BYTES;
  }
  __device__ __forceinline__ u32x4_t read(uint32_t slot) const {
    return *(__attribute__((address_space(3))) u32x4_t *)(uintptr_t)(ring_lane + slot * SP_QUAD_BYTES);
  }
  // Records from batch `first` (counted over all streams) on; the first two quads are asked for.
  __device__ __forceinline__ void begin(const uint32_t *recs, uint32_t first, uint32_t ring_at, uint32_t tile_at, int lane) {
    next = (const char *)recs + (uint64_t)(first / SP_QUAD) * SP_QUAD_BYTES - ring_at;
    ring = ring_at;
    ring_lane = ring_at + (uint32_t)lane * 16;
    at = first % SP_QUAD;
    col = tile_at + (uint32_t)(lane & 3) * 8;
    row_bit = 0x00010001u << (lane & 15);
    ask(0);
    ask(1);
  }
  // They have arrived: the state at which the code of a stage takes batches at places 0 .. 3 up.
  __device__ __forceinline__ void begun() {
    const u32x4_t w = read(0), v = read(1);
    asm volatile("" ::"v"(w), "v"(v));     // the slots have been read
    ask(0);
    words = __builtin_shufflevector(w, v, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // The stage's batches, and the wavefront's loads of the tile that comes next.  It has arrived when this returns.
  template <typename T, typename Fill> __device__ __forceinline__ void stage(SpSums &acc, uint2 c, Fill tile) {
    uint32_t n, m0, since;
    // (uniform, which the compiler does not see everywhere)
    at = __builtin_amdgcn_readfirstlane(at);
    uint64_t quad = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)(uintptr_t)next >> 32)) << 32) |
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint64_t)(uintptr_t)next);
#define SP_STAGE_ASM(M, FILL, ...)                                                                                                 \
    asm volatile(SP_STAGE(M, FILL)                                                                                                 \
                 : "+{v[0:31]}"(acc.lo), "+{v[32:63]}"(acc.hi), "+{v[112:119]}"(words), "+{s[40:41]}"(quad), [at] "+s"(at),         \
                   [since] "=&s"(since), [n] "=&s"(n), "=&{m0}"(m0)                                                                 \
                 : [cx] "s"(c.x), [cy] "s"(c.y), [ring] "s"(ring), [ones] "s"(0x00010001u), [row_bit] "v"(row_bit),                 \
                   [col] "v"(col), [ring_lane] "v"(ring_lane) __VA_ARGS__                                                          \
                 : "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79",  \
                   "v80", "v81", "v82", "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95",  \
                   "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109",      \
                   "scc", "memory")
#define SP_FILL_FROM , [from0] "s"(tile.from), [from1] "s"(tile.from + 64), [to] "s"(tile.to), [off0] "v"(tile.off0), [off1] "v"(tile.off1)
    constexpr bool bf16 = std::is_same<T, bf16_t>::value, fill = std::is_same<Fill, SpFill>::value;
    if constexpr (bf16 && fill) SP_STAGE_ASM("v_mfma_f32_16x16x32_bf16", SP_FILL_IF, SP_FILL_FROM);
    else if constexpr (fill) SP_STAGE_ASM("v_mfma_f32_16x16x32_f16", SP_FILL_IF, SP_FILL_FROM);
    else if constexpr (bf16) SP_STAGE_ASM("v_mfma_f32_16x16x32_bf16", SP_FILL_NONE);
    else SP_STAGE_ASM("v_mfma_f32_16x16x32_f16", SP_FILL_NONE);
#undef SP_FILL_FROM
#undef SP_STAGE_ASM
    next = (const char *)(uintptr_t)quad;
  }
};
