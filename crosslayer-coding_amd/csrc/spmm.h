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
//   y = 3   half of where their tile rows begin in LDS: entry 8 q + x low, entry 8 q + 4 + x high
// - every lane finds what it needs in its own row of 16 lanes, one DPP operand away, so that a record costs one dword of
// LDS traffic per lane beside the eight transposing reads (broadcasting it with two 16-byte reads instead: five vector
// instructions fewer, but a quarter more LDS time per batch).
constexpr int SP_REC_WORDS = 64;

// A tile lies in LDS as two halves of 32 columns, 64 bytes per row; the two 32-byte pieces of a row are exchanged in
// every other group of four rows, so that one piece of eight consecutive rows covers all banks.  Column piece n of a row
// is then at place ^ 32 (n & 1), plus half a tile for n >= 2: one exclusive-or for two reads, the rest in their offsets.
// Which of the two tile buffers a stage uses is known when the records are made and is part of the place.
constexpr int SP_HALF_BYTES = SP_TILE_BYTES / 2;
__host__ __device__ __forceinline__ uint32_t sp_swap(uint32_t r) { return (r >> 2) & 1u; }
__device__ __forceinline__ uint32_t sp_half_place(uint32_t r, uint32_t buffer) { return (buffer << 15) | (r << 5) | (sp_swap(r) << 4); }

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

template <typename T> struct SpMma;
template <> struct SpMma<bf16_t> {
  typedef __attribute__((ext_vector_type(8))) __bf16 frag_t;
  __device__ static __forceinline__ f32x4v_t run(frag_t a, frag_t b, f32x4v_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct SpMma<f16_t> {
  typedef __attribute__((ext_vector_type(8))) _Float16 frag_t;
  __device__ static __forceinline__ f32x4v_t run(frag_t a, frag_t b, f32x4v_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// One batch in the making.  finish() multiplies it; between two finishes a wavefront works out the next batch's
// addresses, sets its eight reads going and builds its operand of values while they are under way.  Lane = 16 q + i
// supplies entries 8 q .. 8 q + 7 of output row i.
template <typename T> struct SpBatch {
  typedef typename SpMma<T>::frag_t frag_t;
  struct Pair { s16x4_t lo, hi; };
  uint32_t a0, a1;        // where the lane's two rows lie in LDS
  Pair w[4];              // 64 x 32 operand, 16 columns of the tile each
  u32x4_t picked;         // 32 x 16 operand of values

  // `rec`: this lane's word of the record; `col`: where the tiles begin in LDS plus 8 * (lane % 4).  (s_nop: the wait states
  // a DPP operand needs after a write)
  __device__ __forceinline__ void address(uint32_t rec, uint32_t col) {
    uint32_t at;
    asm("s_nop 1\n\tv_mov_b32_dpp %0, %1 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf" : "=v"(at) : "v"(rec));
    asm("v_mad_u32_u16 %0, %1, 2, %2" : "=v"(a0) : "v"(at), "v"(col));
    asm("v_mad_u32_u16 %0, %1, 2, %2 op_sel:[1,0,0,0]" : "=v"(a1) : "v"(at), "v"(col));
  }
  __device__ __forceinline__ void read() {
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      w[n].lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)((a0 ^ (uint32_t)((n & 1) << 5)) + (n >> 1) * SP_HALF_BYTES));
      w[n].hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)((a1 ^ (uint32_t)((n & 1) << 5)) + (n >> 1) * SP_HALF_BYTES));
    }
  }
  // The values of the entries that belong to this lane's output row, zero elsewhere: one-hot & row_bit (bit i of both
  // halves) is non-zero there, and min(.., 1) is a factor.  Written out because the compiler turns the packed minimum
  // and product into twice as many compares and selects.
  __device__ __forceinline__ void pick(uint32_t rec, uint32_t row_bit) {
    uint32_t p0, p1, p2, p3, v;
    asm("s_nop 1\n\t"
        "v_and_b32_dpp %0, %5, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_and_b32_dpp %1, %5, %6 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_and_b32_dpp %2, %5, %6 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_and_b32_dpp %3, %5, %6 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_pk_min_u16 %0, %0, %7\n\t"
        "v_pk_min_u16 %1, %1, %7\n\t"
        "v_pk_mul_lo_u16 %0, %0, %4\n\t"
        "v_mov_b32_dpp %4, %5 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_pk_min_u16 %2, %2, %7\n\t"
        "v_pk_min_u16 %3, %3, %7\n\t"
        "v_pk_mul_lo_u16 %1, %1, %4\n\t"
        "v_mov_b32_dpp %4, %5 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_pk_mul_lo_u16 %2, %2, %4\n\t"
        "v_mov_b32_dpp %4, %5 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_pk_mul_lo_u16 %3, %3, %4"
        : "=&v"(p0), "=&v"(p1), "=&v"(p2), "=&v"(p3), "=&v"(v)
        : "v"(rec), "v"(row_bit), "v"(0x00010001u));
    picked = u32x4_t{p0, p1, p2, p3};
  }
  // acc[n]: columns 16 n .. 16 n + 15 of the tile; lane 16 q + i holds columns 4 q .. 4 q + 3 of output row i
  __device__ __forceinline__ void finish(f32x4v_t (&acc)[4]) {
    const frag_t v = __builtin_bit_cast(frag_t, picked);
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[n] = SpMma<T>::run(__builtin_bit_cast(frag_t, w[n]), v, acc[n]);
  }
};
