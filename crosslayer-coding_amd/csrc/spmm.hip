// Sparse cross-layer decode on the matrix cores (reference clt/models/decoder.py:176-340): decoder rows are gathered
// from LDS tiles instead of from the L2 (spmm.h says why).
//
//   k_rec_count / k_rec_streams / k_rec_fill
//                   survivor list (CSR by token) -> one stream of batches per wavefront of k_decode_tiles, in the order
//                   in which it consumes them: by source, tile of SP_ROWS features, group of 16 tokens
//   k_decode_repair / k_grad_repair
//                   sums that are not finite once more, entry by entry: in the one-hot products an infinity or a NaN in a
//                   tile row reaches all 16 output rows of a batch (0 * inf), here only the rows that refer to it
//   k_decode_tiles  one workgroup per (target, 64 columns, part of the tokens): every tile of every source's decoder
//                   passes through LDS once, the sums stay in registers over all sources and features
//   k_grad_tiles    the transposed product of the backward pass: decoder weight gradients from the same lists by feature,
//                   with the Adam step of the weights taken on the spot
#include "adam.h"
#include "spmm.h"

namespace {

constexpr int DT_WAVES = 16;
constexpr int DT_GPW = 4;                  // groups of 16 output rows per wavefront: 64 accumulators per lane

// How one layer's output rows (tokens of a decode, features of a weight gradient) are dealt out.  Groups
// part * groups_per_part + wave + waves * gi of a part belong to wavefront `wave` of its workgroups; the batches of its
// groups, ordered by (layer, tile, gi), are its stream.
struct SpPlan {
  int tiles, groups, parts, groups_per_part, waves, streams, stages;
  __host__ __device__ __forceinline__ int group(int stream, int gi) const {        // -1: none
    const int part = stream / waves, r = stream % waves + gi * waves, g = part * groups_per_part + r;
    return r < groups_per_part && g < groups ? g : -1;
  }
};

// ---- records ----------------------------------------------------------------------------------------
constexpr int REC_THREADS = 256;
constexpr int REC_MAX_TILES = 512;

// The lists that are regrouped: rows r = layer * Rn + row, columns ascending within a row.
struct RecArgs {
  const int32_t *row_ptr, *col;
  const int32_t *src;      // the entry's value is val[src[j]]; null: val[j]
  const void *val;
  int64_t Rn, L, max_entries;
  uint64_t layer_mask;
  SpPlan p;
  int32_t *start;          // [L * groups][SP_GROUP][tiles + 1] list position where a row's entries of a tile begin
  uint16_t *batches;       // [L * tiles][groups] batches of (layer, tile, group)
  uint2 *counts;           // [streams][stages] the same by stream (sp_stage_counts)
  uint32_t *offset;        // [streams][stages] batches of the stream before the stage
  uint32_t *total;         // [streams] batches of the stream, in whole quads
  uint32_t *recs;
  uint32_t *bad;           // number of groups whose sums are not finite, and which
};

// One workgroup per (group of 16 rows, layer).  Rows are sorted by column, so a row's entries of one tile are a run, found
// by binary search.  A layer outside layer_mask counts as empty.
__global__ __launch_bounds__(REC_THREADS) void k_rec_count(RecArgs A) {
  extern __shared__ int32_t run_lds[];
  if (A.row_ptr[A.L * A.Rn] > A.max_entries) return;      // more entries than the workspace was sized for
  const int g = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, tiles = A.p.tiles;
  const int64_t row0 = (int64_t)g * SP_GROUP, r0 = (int64_t)s * A.Rn + row0;
  const bool on = (A.layer_mask >> s) & 1ull;
  int32_t *out = A.start + ((int64_t)s * A.p.groups + g) * SP_GROUP * (tiles + 1);
  for (int i = tid; i < SP_GROUP * (tiles + 1); i += REC_THREADS) {
    const int tk = i / (tiles + 1), c = i - tk * (tiles + 1);
    int32_t lo = 0;
    if (on && row0 + tk < A.Rn) {
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
  for (int c = tid; c < tiles; c += REC_THREADS) {
    int32_t n = 0;
#pragma unroll
    for (int tk = 0; tk < SP_GROUP; ++tk) n += run_lds[tk * (tiles + 1) + c + 1] - run_lds[tk * (tiles + 1) + c];
    A.batches[((int64_t)s * tiles + c) * A.p.groups + g] = (uint16_t)((n + SP_BATCH - 1) / SP_BATCH);
  }
}

// One wavefront per stream: its batch counts per stage and where each stage begins.
__global__ __launch_bounds__(64) void k_rec_streams(RecArgs A) {
  if (A.row_ptr[A.L * A.Rn] > A.max_entries) return;
  const int stream = blockIdx.x, lane = threadIdx.x;
  uint32_t run = 0;
  for (int st0 = 0; st0 < A.p.stages; st0 += 64) {
    const int st = st0 + lane;
    uint32_t n[DT_GPW], sum = 0;
#pragma unroll
    for (int gi = 0; gi < DT_GPW; ++gi) {
      const int g = A.p.group(stream, gi);
      n[gi] = st < A.p.stages && g >= 0 ? A.batches[(int64_t)st * A.p.groups + g] : 0u;
      sum += n[gi];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(incl, o);
      if (lane >= o) incl += up;
    }
    if (st < A.p.stages) {
      A.offset[(int64_t)stream * A.p.stages + st] = run + incl - sum;
      A.counts[(int64_t)stream * A.p.stages + st] = sp_stage_counts(n[0], n[1], n[2], n[3]);
    }
    run += __shfl(incl, 63);
  }
  if (lane == 0) A.total[stream] = (run + SP_QUAD - 1) / SP_QUAD * SP_QUAD;
  if (stream == 0 && lane == 0) *A.bad = 0u;
}

// The entries of a wavefront whose low three bits equal `mine`: `b0`, `b1`, `b2` are the ballots of the three bits.
__device__ __forceinline__ uint64_t same_class(uint64_t valid, uint64_t b0, uint64_t b1, uint64_t b2, uint32_t mine) {
  return valid & ~(b0 ^ (0ull - (uint64_t)(mine & 1u))) & ~(b1 ^ (0ull - (uint64_t)((mine >> 1) & 1u))) &
         ~(b2 ^ (0ull - (uint64_t)((mine >> 2) & 1u)));
}

// One workgroup per (group, layer) again, a wavefront per tile: its entries become the tile's batches, put together in LDS and
// written out lane by lane.
//
// Where an entry goes decides how fast LDS hands out its row.  The 64 lanes of a transposing read ask for sixteen 32-byte
// pieces, eight rows by each half of the wavefront, and eight rows with different r % 8 cover all banks: 1.06 ns
// per read and CU, against 2.19 with rows in random places (profiles/lds_read_probe.txt).  So the tile's entries are sorted by
// r % 8 - within a class they keep their order by (row, column): the order of every sum is fixed - and dealt out in turn
// to the 4 nb half reads of its nb batches: a half read then meets a class twice only if the class has more than 4 nb
// entries.  A place that stays empty refers to the half read's first row, which costs no bank of its own.
// (L = 12, d = 768, F = 24576, 4096 tokens, 200 survivors per token, bf16: this kernel 213 -> 158 us against entries in the
// order of the lists, row by row through a window of 128 batches, k_decode_tiles 3.33 -> 3.17 ms; L = 24, d = 1024, F = 32768:
// 433 -> 266 us, 15.77 -> 15.59 ms.  Bound by the chain of a tile's steps in each wavefront.  Tiles with thousands of entries, L
// = 2, 4096 tokens: 176 us where 16 tokens fire all of 512 neighbouring features, 440 in the gradients of 16 that always fire; with
// all entries once per window 1614 and 4236.)
constexpr int REC_WINDOW = 8;                              // batches a wavefront puts together in LDS
template <typename T> __global__ __launch_bounds__(REC_THREADS) void k_rec_fill(RecArgs A) {
  extern __shared__ int32_t fill_lds[];
  const int g = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, tiles = A.p.tiles, lane = tid & 63, wave = tid >> 6;
  if (A.row_ptr[A.L * A.Rn] > A.max_entries) return;
  if (!((A.layer_mask >> s) & 1ull)) return;
  int32_t *start = fill_lds;                               // [SP_GROUP][tiles + 1]
  uint32_t *dest = (uint32_t *)(start + SP_GROUP * (tiles + 1));       // [tiles] the tile's first batch among all of the stream
  uint32_t *win = dest + tiles + wave * (REC_WINDOW * SP_REC_WORDS);   // this wavefront's batches
  const int32_t *src = A.start + ((int64_t)s * A.p.groups + g) * SP_GROUP * (tiles + 1);
  for (int i = tid; i < SP_GROUP * (tiles + 1); i += REC_THREADS) start[i] = src[i];
  const int part = g / A.p.groups_per_part, r = g - part * A.p.groups_per_part;
  const int stream = part * A.p.waves + r % A.p.waves, gi = r / A.p.waves;
  for (int c = tid; c < tiles; c += REC_THREADS) {
    const int64_t at = (int64_t)stream * A.p.stages + (int64_t)s * tiles + c;
    uint32_t d = A.offset[at];
    const uint32_t before = A.counts[at].x;                // (of groups before one that has batches, all are counted)
    for (int j = 0; j < gi; ++j) d += (before >> (10 * j)) & 1023u;
    dest[c] = d;
  }
  const uint32_t base = stream_first(A.total, stream, lane);
  __syncthreads();
  for (int c = wave; c < tiles; c += REC_THREADS / 64) {
    // row t's run: entries run_at + [run_off, ..) of the tile's, laid end to end
    const int t16 = lane & 15;
    const int32_t run_begin = start[t16 * (tiles + 1) + c];
    int32_t run_off = start[t16 * (tiles + 1) + c + 1] - run_begin;
    const int32_t len = run_off;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const int32_t up = __shfl_up(run_off, o, 16);
      if (t16 >= o) run_off += up;
    }
    const int32_t n = __builtin_amdgcn_readlane(run_off, 15);
    if (n == 0) continue;
    run_off -= len;
    const int32_t run_at = run_begin - run_off;
    const int32_t nb = (n + SP_BATCH - 1) / SP_BATCH, halves = 4 * nb;
    const uint32_t magic = 0xFFFFFFFFu / (uint32_t)halves + 1u;          // p / halves = (p * magic) >> 32 for p, halves < 2^16
    // the i-th entry: its row, place in the list and tile row
    auto entry = [&](int32_t i, int &tk, int32_t &j) {
      tk = 0;
#pragma unroll
      for (int t = 1; t < SP_GROUP; ++t) tk += i >= __builtin_amdgcn_readlane(run_off, t) ? 1 : 0;
      j = __shfl(run_at, tk) + i;
    };
    uint32_t first = 0;                                    // lane l: entries of class l % 8, then where the class begins
    for (int32_t i0 = 0; i0 < n; i0 += 64) {
      int tk;
      int32_t j;
      const bool on = i0 + lane < n;
      entry(on ? i0 + lane : n - 1, tk, j);
      const uint32_t cls = (uint32_t)A.col[j];
      const uint64_t v = __ballot(on), b0 = __ballot(cls & 1u), b1 = __ballot(cls & 2u), b2 = __ballot(cls & 4u);
      first += (uint32_t)__popcll(same_class(v, b0, b1, b2, (uint32_t)lane));
    }
    {
      const uint32_t mine = first;
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) {
        const uint32_t up = __shfl_up(first, o, 8);
        if ((lane & 7) >= o) first += up;
      }
      first -= mine;
    }
    // all entries once more, to their places in the records: half_of(batch of the tile, half word of the batch)
    auto fill = [&](auto half_of) {
      uint32_t next = first;
      for (int32_t i0 = 0; i0 < n; i0 += 64) {
        int tk;
        int32_t j;
        const bool on = i0 + lane < n;
        entry(on ? i0 + lane : n - 1, tk, j);
        const uint32_t f = (uint32_t)A.col[j], cls = f & 7u;
        const uint64_t v = __ballot(on), b0 = __ballot(cls & 1u), b1 = __ballot(cls & 2u), b2 = __ballot(cls & 4u);
        const uint64_t same = same_class(v, b0, b1, b2, cls);
        const uint32_t p = __shfl(next, (int)cls) + __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
        next += (uint32_t)__popcll(same_class(v, b0, b1, b2, (uint32_t)lane));
        const uint32_t slot = __umulhi(p, magic), h = p - slot * (uint32_t)halves;
        const int32_t b = (int32_t)(h >> 2);
        if (!on) continue;
        // half read h % 4 of batch h / 4: h & 1 the half of the wavefront, h & 2 the second four entries of its lane quartets
        const uint32_t side = (h & 1u) * 64;
        auto place = [&](uint32_t sl, uint16_t at) {
          *half_of(b, side + (sl >> 2) * 32 + (4 * (sl & 3u) + 3) * 2 + ((h >> 1) & 1u)) = at;
        };
        const uint32_t k = (slot & 3u) + ((h & 2u) << 1), x = side + (slot >> 2) * 32 + 8 * (k >> 1) + (k & 1u);
        *half_of(b, x) = (uint16_t)Elem<T>::raw(((const T *)A.val)[A.src ? A.src[j] : j]);
        *half_of(b, x + 2) = (uint16_t)(1u << tk);
        const uint16_t at = (uint16_t)sp_place(f - (uint32_t)c * SP_ROWS);
        place(slot, at);
        if (slot == 0)                                     // the places of this half read that stay empty
          for (uint32_t sl = __umulhi((uint32_t)n - 1u - p, magic) + 1u; sl < 8u; ++sl) place(sl, at);
      }
    };
    const uint64_t b0 = (uint64_t)base + dest[c];
    if (nb <= REC_WINDOW) {
      for (int32_t b = 0; b < nb; ++b) win[b * SP_REC_WORDS + lane] = 0u;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      fill([&](int32_t b, uint32_t i) { return (uint16_t *)win + b * (2 * SP_REC_WORDS) + i; });
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int32_t b = 0; b < nb; ++b) A.recs[sp_rec_word(b0 + b, lane)] = win[b * SP_REC_WORDS + lane];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
      // more than the window holds - up to 256, where 16 features fire on most tokens: put together where they are to lie, two
      // bytes at a time, rather than all entries once per window
      for (int32_t b = 0; b < nb; ++b) A.recs[sp_rec_word(b0 + b, lane)] = 0u;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the zeros have arrived
      fill([&](int32_t b, uint32_t i) { return (uint16_t *)(A.recs + sp_rec_word(b0 + b, i >> 1)) + (i & 1u); });
    }
  }
}

// ---- decode -----------------------------------------------------------------------------------------
struct TileArgs {
  SpPlan p;
  const uint2 *counts;
  const uint32_t *total;
  const uint32_t *recs;
  const void *wp;
  const float *bias_sum, *skip_add;
  void *out;
  const int32_t *list_total;               // survivors of the batch
  const int32_t *row_ptr, *col;
  const void *val;
  uint32_t *bad;
  int64_t max_entries, Tn, d, F, L, pitch;
  uint64_t src_mask;
  int tying, t_begin, t_end, out_f32, col_parts;
};

constexpr int DT_FILLS = SP_ROWS / 8 / DT_WAVES;           // direct-to-LDS loads of a tile per wavefront
constexpr int DT_LDS = 2 * SP_TILE_BYTES + DT_WAVES * SP_RING_BYTES;
static_assert(DT_FILLS == 4, "the wait counts here and in SP_RING_READ are written out");

// Whether a wavefront's sums of a group (16 rows from row0 on, of n rows) are all finite; if not, the group goes on the list.
__device__ __forceinline__ bool sums_finite(const f32x4v_t (&acc)[4], bool row_on, uint32_t *bad, uint32_t item) {
  float z = 0.0f;
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int q = 0; q < 4; ++q) z = fmaf(acc[n][q], 0.0f, z);
  if (ballot64(row_on && z != z) == 0) return true;
  if (lane_id() == 0) bad[1 + atomicAdd(bad, 1u)] = item;
  return false;
}

// Two tiles of 512 features x 64 columns in LDS, one being multiplied while the other comes in.  Each wavefront owns four
// groups of 16 tokens and consumes its stream of batches through a ring of two quads of records in LDS: the vector memory path
// returns in order, so a record waits behind whatever tile lines were asked for before it, and the seven batches between a
// quad's request and its use cover that.  Workgroups that share a decoder tile (the parts of the tokens) follow each other on one
// XCD, so that one of them brings it from HBM and the others find it in the L2.
//
// L = 12, d = 768, F = 24576, 4096 tokens, 200 survivors per token, untied, bf16: 2.82 ms (98.6 GB of gathered rows, 35
// TB/s) and 0.19 ms for the records, against 6.45 ms of the gather from the L2s; L = 24, d = 1024, F = 32768: 14.4 and 0.39
// against 34.2 ms.  A record at a time and one batch in the making took 3.10 and 15.5 ms.  It is 5.6 M cycles of a clock that the
// power limit holds at 1.97 GHz (6.3 M at 2.09 before); in those vector instructions issue 53 % of the time, LDS is active 45 %,
// the matrix cores 33 %, and the wavefronts wait 43 % of theirs, most of it at the barrier for the one with the heaviest
// tokens (decode_tiles_c1_lds_counters.txt; with equal lists 2.65 ms).  Without batches the tiles alone take 1.65 ms to come in.
// Measured and dropped: reads and products of a step interleaved, or the values' operand first (within 1 %: no single step binds);
// heavy wavefronts at a higher wave priority (the same); a wavefront of its own for the fills (fifteen share 64 groups badly:
// 3.98 ms); fewer lines on their way (4.5 ms: the fills are latency-bound); every parts-th line of the tile after next brought
// into the L2 early (3.46 ms: the early loads block the records just as well).
template <typename T>
__global__ __launch_bounds__(DT_WAVES * 64) void k_decode_tiles(TileArgs A) {
  extern __shared__ __attribute__((aligned(128))) char tile_lds[];
  if (*A.list_total > A.max_entries) return;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int pair = (seq / A.p.parts) * 8 + xcd, part = seq % A.p.parts;
  if (pair >= (A.t_end - A.t_begin) * A.col_parts) return;
  const int t = A.t_end - 1 - pair / A.col_parts, cp = pair % A.col_parts;      // longest first
  const uint64_t mask = A.src_mask & ((2ull << t) - 1ull);
  const int n_stages = __popcll(mask) * A.p.tiles;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)tile_lds;
  const int stream = part * DT_WAVES + wave;

  // This wavefront's share of a tile: 32 rows, sixteen at a time and one half of the columns at a time, 16 bytes of row
  // lane / 4 per lane; which 16 bytes a lane brings is what exchanges the pieces.  (Both halves of a line are asked for
  // one after the other: the second hits the L1.)
  const uint32_t pitch_b = (uint32_t)(A.pitch * (int64_t)sizeof(T));
  // Rows past the matrix, which nobody refers to, are read as its last one.
  const uint32_t off_a = (uint32_t)(wave * 32 + (lane >> 2)) * pitch_b + ((((((uint32_t)lane & 3) >> 1) ^ sp_swap(lane >> 2)) << 5) | ((lane & 1) << 4));
  const uint32_t off_b = off_a + 16 * pitch_b;
  auto last_row = [&](int rows) { return (uint32_t)((rows < SP_ROWS ? rows : SP_ROWS) - 1) * pitch_b + 48u; };

  auto tile_at = [&](int s) {
    return (const char *)A.wp + sp_slot(A.tying, s, t, A.L) * A.F * (int64_t)pitch_b + (int64_t)cp * 128;
  };

  SpSums acc;
  acc.clear();
  if (n_stages > 0) {
    SpStream batches;
    batches.begin(A.recs, __builtin_amdgcn_readfirstlane(stream_first(A.total, stream, lane)), lds0 + 2 * SP_TILE_BYTES + (uint32_t)wave * SP_RING_BYTES, lds0, lane);
    // the next tile to bring in: where it begins and how many rows of the matrix are left from there on
    uint64_t m = mask;
    int s = __ffsll((unsigned long long)m) - 1, c = 0, rows = (int)A.F;
    const char *tile = tile_at(s);
    const uint32_t tile_step = SP_ROWS * pitch_b, lds_share = lds0 + (uint32_t)wave * 2048;
    {
      const uint32_t last = last_row(rows);
#pragma unroll
      for (int i = 0; i < DT_FILLS; ++i) {
        const uint32_t off = i >> 1 ? off_b : off_a;
        sp_fill16(tile + (i & 1) * 64, off < last ? off : last, lds_share + (uint32_t)((i >> 1) * 1024 + (i & 1) * SP_HALF_BYTES));
      }
    }
    const auto stream_counts = (const __attribute__((address_space(4))) uint2 *)(uintptr_t)A.counts + (int64_t)stream * A.p.stages;
    auto counts = stream_counts + s * A.p.tiles;
    uint2 cnt = make_uint2(counts->x, counts->y);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    batches.begun();
    asm volatile("" ::"v"(batches.words));
    for (int st = 0; st < n_stages; ++st) {
      uint32_t to = SP_NO_TILE;                            // where this wavefront's share of the next tile goes, if there is one
      if (st + 1 < n_stages) {
        tile += tile_step;
        rows -= SP_ROWS;
        ++counts;
        if (++c == A.p.tiles) {
          c = 0;
          m &= m - 1;
          s = __ffsll((unsigned long long)m) - 1;
          tile = tile_at(s);
          rows = (int)A.F;
          counts = stream_counts + s * A.p.tiles;
        }
        to = (lds_share ^ (uint32_t)((st & 1) ^ 1) * SP_TILE_BYTES);
      }
      const uint32_t last = last_row(rows);
      const uint2 cnt_next = make_uint2(counts->x, counts->y);
      const uint32_t off0 = off_a < last ? off_a : last, off1 = off_b < last ? off_b : last;
      asm volatile("" ::"v"(off0), "v"(off1) : "memory");
      __builtin_amdgcn_s_barrier();                        // tile st is complete, and nobody reads the other one any more
      asm volatile("" ::: "memory");
      batches.stage<T>(acc, cnt, SpFill{tile, off0, off1, to});
      batches.col += st & 1 ? -SP_TILE_BYTES : SP_TILE_BYTES;
      cnt = cnt_next;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may be on its way into LDS when the workgroup ends
  }

#pragma unroll
  for (int gi = 0; gi < DT_GPW; ++gi) {
    const int g = A.p.group(stream, gi);
    const int64_t tok = (int64_t)g * SP_GROUP + (lane & 15);
    if (g < 0) continue;
    f32x4v_t sum[4];
    acc.get(gi, sum);
    if (!sums_finite(sum, tok < A.Tn, A.bad, (uint32_t)(((t - A.t_begin) * A.p.groups + g) * A.col_parts + cp)) || tok >= A.Tn) continue;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int64_t o = (int64_t)cp * SP_COLS + n * 16 + (lane >> 4) * 4;
      f32x4v_t a = sum[n];
      const int64_t at = ((int64_t)t * A.Tn + tok) * A.d + o;
      if (A.bias_sum) a += *reinterpret_cast<const f32x4v_t *>(A.bias_sum + (int64_t)t * A.d + o);
      if (A.skip_add) a += *reinterpret_cast<const f32x4v_t *>(A.skip_add + at);
      if (A.out_f32) *reinterpret_cast<f32x4v_t *>((float *)A.out + at) = a;
      else *reinterpret_cast<uint2 *>((uint16_t *)A.out + at) = make_uint2(pack_pair<T>(a[0], a[1]), pack_pair<T>(a[2], a[3]));
    }
  }
}

// The listed groups (16 tokens x 64 columns of a target): a thread sums 4 columns of a token over its survivors.
template <typename T> __global__ __launch_bounds__(256) void k_decode_repair(TileArgs A) {
  if (*A.list_total > A.max_entries) return;
  const uint32_t n = *A.bad;
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t item = A.bad[1 + i], cp = item % A.col_parts, g = item / A.col_parts % A.p.groups;
    const int64_t t = A.t_begin + item / A.col_parts / A.p.groups, tok = (int64_t)g * SP_GROUP + (threadIdx.x >> 4);
    if (tok >= A.Tn) continue;
    const int64_t o = (int64_t)cp * SP_COLS + (threadIdx.x & 15) * 4, at = (t * A.Tn + tok) * A.d + o;
    f32x4v_t a{0.f, 0.f, 0.f, 0.f};
    for (int64_t s = 0; s <= t; ++s) {
      if (!((A.src_mask >> s) & 1ull)) continue;
      const T *w = (const T *)A.wp + sp_slot(A.tying, s, t, A.L) * A.F * A.pitch + o;
      for (int32_t j = A.row_ptr[s * A.Tn + tok]; j < A.row_ptr[s * A.Tn + tok + 1]; ++j) {
        const uint2 raw = *reinterpret_cast<const uint2 *>(w + (int64_t)A.col[j] * A.pitch);
        const float v = Elem<T>::to_f32(((const T *)A.val)[j]);
        float x[4];
        unpack_pair<T>(raw.x, x[0], x[1]);
        unpack_pair<T>(raw.y, x[2], x[3]);
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = fmaf(v, x[q], a[q]);
      }
    }
    if (A.bias_sum) a += *reinterpret_cast<const f32x4v_t *>(A.bias_sum + t * A.d + o);
    if (A.skip_add) a += *reinterpret_cast<const f32x4v_t *>(A.skip_add + at);
    if (A.out_f32) *reinterpret_cast<f32x4v_t *>((float *)A.out + at) = a;
    else *reinterpret_cast<uint2 *>((uint16_t *)A.out + at) = make_uint2(pack_pair<T>(a[0], a[1]), pack_pair<T>(a[2], a[3]));
  }
}

// ---- decoder weight gradient (and Adam) ---------------------------------------------------------------
// dW[s->t][f][:] = sum over the tokens of feature f of value * g[t][token][:]: the same product with features in the
// place of tokens - 16 features per group, tiles of 512 tokens x 64 columns of g[t].
constexpr int GT_WAVES = 8;
constexpr int GT_FILLS = SP_ROWS / 8 / GT_WAVES;
constexpr int GT_LDS = SP_TILE_BYTES + GT_WAVES * SP_RING_BYTES;
constexpr int GT_PITCH = SP_COLS + 4;      // fp32 row pitch of a group's gradient on its way through LDS
static_assert(GT_LDS * 2 <= 160 * 1024 && SP_GROUP * GT_PITCH * 4 * GT_WAVES <= SP_TILE_BYTES, "two workgroups per CU");

struct GradArgs {
  SpPlan p;
  const uint2 *counts;
  const uint32_t *offset, *total, *recs;
  const void *g;             // [L][T][d]
  void *w;                   // packed decoders (GT_ADAM)
  float *m, *v;              // moments
  float *out;                // the gradient as fp32 [n_dec][F][d] (GT_ROWS)
  void *const *params;       // [n_dec] where each decoder's gradient goes, [d][F] of T (GT_PARAM)
  int64_t Tn, d, F, L, pitch, max_entries;
  int64_t m_row, m_cols, m_dec;   // moments: elements between rows, between column parts of 64 and between decoders
  const int32_t *list_total, *list_ptr, *list_tok, *list_src;
  const void *val;
  uint32_t *bad;
  int col_parts, items;      // items of one (source, target) pair per XCD
  AdamCoef adam;
};

// What becomes of the sums: an Adam step of the weights, fp32 rows by feature, or the parameters' own layout and type.
enum GradOut { GT_ADAM, GT_ROWS, GT_PARAM };
constexpr int GT_PARAM_PITCH = GT_WAVES * DT_GPW * SP_GROUP + 8;      // a column's features on their way through LDS
static_assert(SP_COLS * GT_PARAM_PITCH * 2 <= GT_LDS, "one workgroup's sums in 16 bits");

// One workgroup per (source, target, 64 columns, part of the features): eight wavefronts, four groups of 16 features each.
// The weights and moments stream through once (20 bytes per weight, nothing else from HBM), which bounds the kernel; so
// two workgroups share a CU (80 KB of LDS each, one tile buffer) and one's products run under the other's streaming.
// A group's sums go through LDS so that 16 lanes read and write 256 contiguous bytes of the moments.  An XCD takes one
// eighth of the features of a pair with all its column parts: the batches' records are read from its L2 by all of them.
//
// GT_PARAM: all sums of a workgroup meet in LDS, from where a column's 512 features go out as 1 KB (L = 6, d = 512, F = 16384, 2048
// tokens, 21 decoders: 242 us, against 233 us for fp32 rows and 298 us for 21 passes that round and transpose them).
template <typename T, GradOut OUT>
__global__ __launch_bounds__(GT_WAVES * 64, 4) void k_grad_tiles(GradArgs A) {
  extern __shared__ __attribute__((aligned(128))) char grad_lds[];
  if (*A.list_total > A.max_entries) return;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int slot = seq / A.items, item = xcd * A.items + seq % A.items;
  if (item >= A.p.parts * A.col_parts) return;
  const int part = item / A.col_parts, cp = item % A.col_parts;
  // decoder `slot` of "0->0", "0->1", ..: source s, target t
  int s = 0, t = slot;
  while (t >= (int)A.L - s) { t -= (int)A.L - s; ++s; }
  t += s;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)grad_lds;
  const int stream = part * GT_WAVES + wave;

  const uint32_t pitch_b = (uint32_t)(A.d * (int64_t)sizeof(T));
  const uint32_t off_a = (uint32_t)(wave * 64 + (lane >> 2)) * pitch_b + ((((((uint32_t)lane & 3) >> 1) ^ sp_swap(lane >> 2)) << 5) | ((lane & 1) << 4));
  auto fill = [&](const char *src, int rows) {             // as in k_decode_tiles
    const uint32_t last = (uint32_t)((rows < SP_ROWS ? rows : SP_ROWS) - 1) * pitch_b + 48u;
#pragma unroll
    for (int i = 0; i < GT_FILLS; ++i) {
      const uint32_t off = off_a + (uint32_t)(i >> 1) * 16 * pitch_b;
      sp_fill16(src + (i & 1) * 64, off < last ? off : last, lds0 + (uint32_t)(wave * 4096 + (i >> 1) * 1024 + (i & 1) * SP_HALF_BYTES));
    }
  };

  SpSums acc;
  acc.clear();
  {
    const int stage0 = s * A.p.tiles;
    SpStream batches;
    batches.begin(A.recs, __builtin_amdgcn_readfirstlane(stream_first(A.total, stream, lane) + A.offset[(int64_t)stream * A.p.stages + stage0]),
                  lds0 + SP_TILE_BYTES + (uint32_t)wave * SP_RING_BYTES, lds0, lane);
    const auto counts = (const __attribute__((address_space(4))) uint2 *)(uintptr_t)A.counts + (int64_t)stream * A.p.stages + stage0;
    const char *tile = (const char *)A.g + (int64_t)t * A.Tn * (int64_t)pitch_b + (int64_t)cp * 128;
    fill(tile, (int)A.Tn);
    uint2 cnt = make_uint2(counts->x, counts->y);
    asm volatile("s_waitcnt vmcnt(0)" ::"s"(cnt.x), "s"(cnt.y) : "memory");
    batches.begun();
    int rows = (int)A.Tn;
    for (int st = 0; st < A.p.tiles; ++st) {
      if (st > 0) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();                      // nobody reads the last tile any more
        asm volatile("" ::: "memory");
        tile += SP_ROWS * pitch_b;
        rows -= SP_ROWS;
        fill(tile, rows);
        cnt = make_uint2(counts[st].x, counts[st].y);      // (arrives before the tile does)
        asm volatile("s_waitcnt vmcnt(0)" ::"s"(cnt.x), "s"(cnt.y) : "memory");
      }
      asm volatile("" ::"v"(batches.words) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      batches.stage<T>(acc, cnt, SpNoFill{});              // (there is one buffer: no tile comes in meanwhile)
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                          // the tile's LDS is free
    asm volatile("" ::: "memory");
  }

  if constexpr (OUT == GT_PARAM) {
    uint16_t *const cols = (uint16_t *)grad_lds;
#pragma unroll
    for (int gi = 0; gi < DT_GPW; ++gi) {
      const int g = A.p.group(stream, gi);
      if (g < 0) continue;
      f32x4v_t sum[4];
      acc.get(gi, sum);
      sums_finite(sum, (int64_t)g * SP_GROUP + (lane & 15) < A.F, A.bad, (uint32_t)((slot * A.p.groups + g) * A.col_parts + cp));
      uint16_t *const at = cols + (lane >> 4) * 4 * GT_PARAM_PITCH + (wave + gi * GT_WAVES) * SP_GROUP + (lane & 15);
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int k = 0; k < 4; ++k) at[(n * 16 + k) * GT_PARAM_PITCH] = (uint16_t)Elem<T>::raw(Elem<T>::from_f32(sum[n][k]));
    }
    __syncthreads();
    const int64_t f = (int64_t)part * A.p.groups_per_part * SP_GROUP + lane * 8;
    if (lane * 8 < A.p.groups_per_part * SP_GROUP && f < A.F) {      // (F is a multiple of eight)
      T *const out = (T *)A.params[slot] + (int64_t)cp * SP_COLS * A.F + f;
#pragma unroll
      for (int c = wave; c < SP_COLS; c += GT_WAVES)
        *reinterpret_cast<uint4 *>(out + c * A.F) = *reinterpret_cast<const uint4 *>(cols + c * GT_PARAM_PITCH + lane * 8);
    }
    return;
  }
  float *const mine = (float *)(grad_lds + wave * (SP_GROUP * GT_PITCH * 4));
#pragma unroll
  for (int gi = 0; gi < DT_GPW; ++gi) {
    const int g = A.p.group(stream, gi);
    if (g < 0) break;
    f32x4v_t sum[4];
    acc.get(gi, sum);
    if (!sums_finite(sum, (int64_t)g * SP_GROUP + (lane & 15) < A.F, A.bad, (uint32_t)((slot * A.p.groups + g) * A.col_parts + cp))) continue;
    // rows of 64 columns: lane 16 r + c takes columns 4 c .. 4 c + 3 of rows r, r + 4, r + 8, r + 12
    const int c4 = (lane & 15) * 4;
    const int64_t f0 = (int64_t)g * SP_GROUP + (lane >> 4);
    float *const m_at = A.m + slot * A.m_dec + (int64_t)cp * A.m_cols + f0 * A.m_row + c4;
    float *const v_at = A.v + slot * A.m_dec + (int64_t)cp * A.m_cols + f0 * A.m_row + c4;
    uint16_t *const w_at = (uint16_t *)A.w + ((int64_t)slot * A.F + f0) * A.pitch + (int64_t)cp * SP_COLS + c4;
    f32x4v_t mm[4], vv[4];
    uint2 ww[4];
    if constexpr (OUT == GT_ADAM) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t o = f0 + 4 * i < A.F ? 4 * i : -(f0 - (f0 < A.F ? f0 : 0));      // past the last feature: a row that exists
        mm[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4v_t *>(m_at + o * A.m_row));
        vv[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4v_t *>(v_at + o * A.m_row));
        ww[i] = *reinterpret_cast<const uint2 *>(w_at + o * A.pitch);
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n)
      *reinterpret_cast<f32x4v_t *>(mine + (lane & 15) * GT_PITCH + n * 16 + (lane >> 4) * 4) = sum[n];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4v_t gr = *reinterpret_cast<const f32x4v_t *>(mine + ((lane >> 4) + 4 * i) * GT_PITCH + c4);
      if (f0 + 4 * i >= A.F) continue;
      if constexpr (OUT == GT_ADAM) {
        float p[4];
        unpack_pair<T>(ww[i].x, p[0], p[1]);
        unpack_pair<T>(ww[i].y, p[2], p[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float m1 = mm[i][k], v1 = vv[i][k];
          p[k] = adam_update(p[k], gr[k], m1, v1, A.adam);
          mm[i][k] = m1;
          vv[i][k] = v1;
        }
        __builtin_nontemporal_store(mm[i], reinterpret_cast<f32x4v_t *>(m_at + 4 * i * A.m_row));
        __builtin_nontemporal_store(vv[i], reinterpret_cast<f32x4v_t *>(v_at + 4 * i * A.m_row));
        *reinterpret_cast<uint2 *>(w_at + 4 * i * A.pitch) = make_uint2(pack_pair<T>(p[0], p[1]), pack_pair<T>(p[2], p[3]));
      } else {
        __builtin_nontemporal_store(gr, reinterpret_cast<f32x4v_t *>(A.out + ((int64_t)slot * A.F + f0 + 4 * i) * A.d + (int64_t)cp * SP_COLS + c4));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");    // read before the next group's sums are written
  }
}

// The listed groups (16 features x 64 columns of a decoder): a thread sums 4 columns of a feature over its list and steps.
template <typename T, GradOut OUT> __global__ __launch_bounds__(256) void k_grad_repair(GradArgs A) {
  if (*A.list_total > A.max_entries) return;
  const uint32_t n = *A.bad;
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t item = A.bad[1 + i], cp = item % A.col_parts, g = item / A.col_parts % A.p.groups;
    const int64_t slot = item / A.col_parts / A.p.groups, f = (int64_t)g * SP_GROUP + (threadIdx.x >> 4);
    if (f >= A.F) continue;
    int64_t s = 0, t = slot;
    while (t >= A.L - s) { t -= A.L - s; ++s; }
    t += s;
    const int c4 = (threadIdx.x & 15) * 4;
    const T *g_at = (const T *)A.g + t * A.Tn * A.d + (int64_t)cp * SP_COLS + c4;
    float gr[4] = {0.f, 0.f, 0.f, 0.f};
    for (int32_t j = A.list_ptr[s * A.F + f]; j < A.list_ptr[s * A.F + f + 1]; ++j) {
      const uint2 raw = *reinterpret_cast<const uint2 *>(g_at + (int64_t)A.list_tok[j] * A.d);
      const float v = Elem<T>::to_f32(((const T *)A.val)[A.list_src[j]]);
      float x[4];
      unpack_pair<T>(raw.x, x[0], x[1]);
      unpack_pair<T>(raw.y, x[2], x[3]);
#pragma unroll
      for (int q = 0; q < 4; ++q) gr[q] = fmaf(v, x[q], gr[q]);
    }
    if constexpr (OUT == GT_ADAM) {
      const int64_t at = slot * A.m_dec + (int64_t)cp * A.m_cols + f * A.m_row + c4;
      T *w = (T *)A.w + (slot * A.F + f) * A.pitch + (int64_t)cp * SP_COLS + c4;
#pragma unroll
      for (int q = 0; q < 4; ++q) w[q] = Elem<T>::from_f32(adam_update(Elem<T>::to_f32(w[q]), gr[q], A.m[at + q], A.v[at + q], A.adam));
    } else {
      const int64_t c = (int64_t)cp * SP_COLS + c4;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (OUT == GT_ROWS) A.out[(slot * A.F + f) * A.d + c + q] = gr[q];
        else ((T *)A.params[slot])[(c + q) * A.F + f] = Elem<T>::from_f32(gr[q]);
      }
    }
  }
}
constexpr unsigned REPAIR_BLOCKS = 512;

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

struct SpLayout {
  SpPlan p;
  int col_parts;
  int64_t n_batches, n_groups;
  size_t bad, start, batches, counts, offset, total, recs, params, bytes;
};

// `rows` output rows and `cols` tile rows per layer; `per_part` workgroups for every part of the rows; `outputs` times that
// many rows come out
static SpLayout sp_layout(int64_t rows, int64_t cols, int64_t d, int64_t L, int waves, int64_t per_part, int64_t outputs, int64_t max_entries) {
  SpLayout l;
  SpPlan &p = l.p;
  p.tiles = (int)clt_ceil_div(cols, SP_ROWS);
  p.groups = (int)clt_ceil_div(rows, SP_GROUP);
  p.stages = (int)(L * p.tiles);
  p.waves = waves;
  l.col_parts = (int)(d / SP_COLS);
  // as many rows per workgroup as its registers hold, unless that leaves compute units idle
  for (int gpw = DT_GPW; gpw > 0; --gpw) {
    p.parts = (int)clt_ceil_div(p.groups, waves * gpw);
    if ((int64_t)p.parts * l.col_parts * per_part >= 512) break;
  }
  p.groups_per_part = (int)clt_ceil_div(p.groups, p.parts);
  p.streams = p.parts * waves;
  // every (layer, tile, group) may leave its last batch part empty, and every stream its last quad
  l.n_batches = max_entries / SP_BATCH + (int64_t)p.stages * p.groups;
  const int64_t rec_batches = l.n_batches + (int64_t)(SP_QUAD - 1) * p.streams + SP_PAST_END;
  size_t at = 0;
  auto take = [&](size_t n) { const size_t here = at; at += align256(n); return here; };
  l.start = take(sizeof(int32_t) * (size_t)L * p.groups * SP_GROUP * (p.tiles + 1));
  l.batches = take(sizeof(uint16_t) * (size_t)p.stages * p.groups);
  l.counts = take(sizeof(uint2) * (size_t)p.streams * p.stages);
  l.offset = take(sizeof(uint32_t) * (size_t)p.streams * p.stages);
  l.total = take(sizeof(uint32_t) * (size_t)p.streams);
  l.recs = take((size_t)rec_batches * SP_REC_WORDS * 4);
  l.n_groups = outputs * p.groups * l.col_parts;
  l.bad = take(sizeof(uint32_t) * (size_t)(l.n_groups + 1));
  l.params = take(sizeof(void *) * (size_t)outputs);
  l.bytes = at;
  return l;
}

// LDS for the run starts of every tile; 32-bit offsets of rows within a tile; 16-bit batch counts; batches whose records take 4 GB
constexpr int64_t SP_MAX_BATCHES = 0x00FFFFFF;
static bool sp_shape_ok(const SpLayout &l, int64_t row_bytes) {
  return l.p.tiles <= REC_MAX_TILES && l.n_batches <= SP_MAX_BATCHES && row_bytes * SP_ROWS <= 0x7FFFFFFFll && l.p.groups <= 0xFFFF &&
         (int64_t)l.p.stages * l.p.groups <= 0x7FFFFFFFll && l.n_groups <= 0x7FFFFFFFll;
}

static void sp_place_workspace(RecArgs &ra, const SpLayout &l, char *ws) {
  ra.p = l.p;
  ra.start = (int32_t *)(ws + l.start); ra.batches = (uint16_t *)(ws + l.batches); ra.counts = (uint2 *)(ws + l.counts);
  ra.offset = (uint32_t *)(ws + l.offset); ra.total = (uint32_t *)(ws + l.total); ra.recs = (uint32_t *)(ws + l.recs);
  ra.bad = (uint32_t *)(ws + l.bad);
}

template <typename T> static int launch_records(RecArgs ra, hipStream_t stream) {
  const int tiles = ra.p.tiles;
  const size_t count_lds = sizeof(int32_t) * (size_t)SP_GROUP * (tiles + 1);
  const size_t fill_lds = count_lds + sizeof(uint32_t) * ((size_t)tiles + (size_t)REC_THREADS / 64 * REC_WINDOW * SP_REC_WORDS);
  if (hipFuncSetAttribute((const void *)k_rec_fill<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)fill_lds) != hipSuccess)
    return CLT_ERR_LAUNCH;
  const dim3 grid((unsigned)ra.p.groups, (unsigned)ra.L);
  k_rec_count<<<grid, REC_THREADS, count_lds, stream>>>(ra);
  k_rec_streams<<<(unsigned)ra.p.streams, 64, 0, stream>>>(ra);
  k_rec_fill<T><<<grid, REC_THREADS, fill_lds, stream>>>(ra);
  return CLT_OK;
}

static SpLayout tile_layout(int64_t Tn, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t max_entries) {
  return sp_layout(Tn, F, d, L, DT_WAVES, targets, targets, max_entries);
}

template <typename T> static int launch_tiles(RecArgs ra, TileArgs ta, int col_parts, hipStream_t stream) {
  const int code = launch_records<T>(ra, stream);
  if (code != CLT_OK) return code;
  if (hipFuncSetAttribute((const void *)k_decode_tiles<T>, hipFuncAttributeMaxDynamicSharedMemorySize, DT_LDS) != hipSuccess)
    return CLT_ERR_LAUNCH;
  const int64_t pairs = clt_ceil_div((int64_t)(ta.t_end - ta.t_begin) * col_parts, 8) * 8;
  k_decode_tiles<T><<<(unsigned)(pairs * ta.p.parts), DT_WAVES * 64, DT_LDS, stream>>>(ta);
  k_decode_repair<T><<<REPAIR_BLOCKS, 256, 0, stream>>>(ta);
  return clt_check_launch();
}

static SpLayout grad_layout(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries) {
  // (a launch has a workgroup per pair, column part and part of the features: plenty, so the parts are as large as they get)
  return sp_layout(F, T, d, L, GT_WAVES, 1 << 20, L * (L + 1) / 2, entries);
}

// Addresses as kernel arguments, so that nothing on the host has to outlive the call.
constexpr int ADDRESSES = 256;
struct Addresses { void *at[ADDRESSES]; };
__global__ __launch_bounds__(ADDRESSES) void k_set_addresses(Addresses a, int n, void **to) {
  if ((int)threadIdx.x < n) to[threadIdx.x] = a.at[threadIdx.x];
}

// `params`: host array of n_dec addresses (GT_PARAM)
static int launch_grad(GradOut out, const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val, GradArgs a,
                       void *const *params, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  const SpLayout l = grad_layout(a.Tn, a.d, a.F, a.L, a.max_entries);
  if (!sp_shape_ok(l, a.d * 2)) return CLT_ERR_RANGE;
  if (workspace_bytes < l.bytes) return CLT_ERR_WORKSPACE;
  RecArgs ra;
  ra.row_ptr = list_ptr; ra.col = list_tok; ra.src = list_src; ra.val = val; ra.Rn = a.F; ra.L = a.L; ra.max_entries = a.max_entries;
  ra.layer_mask = ~0ull;
  sp_place_workspace(ra, l, (char *)workspace);
  const int code = launch_records<bf16_t>(ra, stream);
  if (code != CLT_OK) return code;
  a.p = l.p; a.counts = ra.counts; a.offset = ra.offset; a.total = ra.total; a.recs = ra.recs;
  a.list_total = list_ptr + a.L * a.F;
  a.list_ptr = list_ptr; a.list_tok = list_tok; a.list_src = list_src; a.val = val; a.bad = ra.bad;
  a.col_parts = l.col_parts;
  a.items = (int)clt_ceil_div((int64_t)l.p.parts * l.col_parts, 8);
  const int64_t blocks = 8 * (int64_t)a.items * (a.L * (a.L + 1) / 2);
  if (blocks > 0x7FFFFFFFll) return CLT_ERR_RANGE;
  const void *k = out == GT_ADAM ? (const void *)k_grad_tiles<bf16_t, GT_ADAM>
                 : out == GT_ROWS ? (const void *)k_grad_tiles<bf16_t, GT_ROWS> : (const void *)k_grad_tiles<bf16_t, GT_PARAM>;
  if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, GT_LDS) != hipSuccess) return CLT_ERR_LAUNCH;
  if (out == GT_ADAM) {
    k_grad_tiles<bf16_t, GT_ADAM><<<(unsigned)blocks, GT_WAVES * 64, GT_LDS, stream>>>(a);
    k_grad_repair<bf16_t, GT_ADAM><<<REPAIR_BLOCKS, 256, 0, stream>>>(a);
  } else if (out == GT_ROWS) {
    k_grad_tiles<bf16_t, GT_ROWS><<<(unsigned)blocks, GT_WAVES * 64, GT_LDS, stream>>>(a);
    k_grad_repair<bf16_t, GT_ROWS><<<REPAIR_BLOCKS, 256, 0, stream>>>(a);
  } else {
    void **const table = (void **)((char *)workspace + l.params);
    const int n_dec = (int)(a.L * (a.L + 1) / 2);
    for (int i0 = 0; i0 < n_dec; i0 += ADDRESSES) {
      Addresses some;
      const int n = n_dec - i0 < ADDRESSES ? n_dec - i0 : ADDRESSES;
      for (int i = 0; i < ADDRESSES; ++i) some.at[i] = i < n ? params[i0 + i] : nullptr;
      k_set_addresses<<<1, ADDRESSES, 0, stream>>>(some, n, table + i0);
    }
    a.params = table;
    k_grad_tiles<bf16_t, GT_PARAM><<<(unsigned)blocks, GT_WAVES * 64, GT_LDS, stream>>>(a);
    k_grad_repair<bf16_t, GT_PARAM><<<REPAIR_BLOCKS, 256, 0, stream>>>(a);
  }
  return clt_check_launch();
}

}  // namespace

// Priced from what it measured (16 bits; 3510 of the shapes of clt_decode_gather_us; off by 12 % in the mean): a stage of the tiles takes
// 1.1 us plus 15 ns per batch, but no less than 64 KB take to come into LDS, 1.7 us from HBM and 0.5 where the targets share a decoder;
// workgroups of unequal length end a quarter of the longest behind the mean, and the longest one bounds a launch of few.  E.g. us, tiles
// / gather: L = 12, d = 768, F = 24576: 2958 / 6769 with 200 per token at T = 4096, 1565 / 2782 at 1024, 1297 / 1440 at 512, 1360 / 846 at
// 256; 1700 / 2703 with 50 at 4096, 1545 / 1642 at 2048; L = 4, d = 512, F = 8192, 1024 x 100: 137 / 238.
double clt_decode_tiles_us(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying, int dtype) {
  const double no = 1e30;
  if ((dtype != CLT_BF16 && dtype != CLT_F16) || (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE)) return no;
  if (T <= 0 || d <= 0 || d % SP_COLS != 0 || F <= 0 || L <= 0 || L > 64 || targets <= 0 || targets > L || entries <= 0) return no;
  const SpLayout l = tile_layout(T, d, F, L, targets, entries);
  if (!sp_shape_ok(l, clt_pitch(d, 2) * 2)) return no;
  const double pairs = 0.5 * targets * (2 * L - targets + 1);
  const double per_batch = (double)entries / ((double)l.p.stages * l.p.groups) / SP_BATCH + 0.15;
  const double stage = 1.09 + l.p.groups_per_part * (per_batch > 1 ? per_batch : 1) * 0.015, fill = tying == CLT_TYING_NONE ? 1.72 : 0.52;
  const double stages = pairs * l.p.tiles * l.col_parts * l.p.parts / 256, longest = (double)L * l.p.tiles;
  const double last = stages + 0.23 * longest > 1.06 * longest ? stages + 0.23 * longest : 1.06 * longest;
  return last * (stage > fill ? stage : fill) + 13 + entries * 1.3e-5;
}

extern "C" int clt_decode_tiles_wanted(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t entries, int tying,
                                       int dtype) {
  const double us = clt_decode_tiles_us(T, d, F, L, targets, entries, tying, dtype);
  return us < 1e30 && us < 0.95 * clt_decode_gather_us(T, d, F, L, targets, entries, tying, dtype);
}

extern "C" int64_t clt_decode_tiles_max_entries(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets) {
  if (T <= 0 || d < SP_COLS || F <= 0 || L <= 0 || targets <= 0) return 0;
  const SpLayout l = tile_layout(T, d, F, L, targets, 0);
  return sp_shape_ok(l, clt_pitch(d, 2) * 2) ? (SP_MAX_BATCHES - l.n_batches) * SP_BATCH + SP_BATCH - 1 : 0;
}

extern "C" size_t clt_decode_tiles_workspace_bytes(int64_t T, int64_t d, int64_t F, int64_t L, int64_t targets, int64_t max_entries) {
  if (T <= 0 || d < SP_COLS || F <= 0 || L <= 0 || targets <= 0 || max_entries < 0) return 0;
  return tile_layout(T, d, F, L, targets, max_entries).bytes;
}

extern "C" int clt_decode_tiles(const int32_t *row_ptr, const int32_t *col, const void *val, const void *w_packed,
                                const float *bias_sum, const float *skip_add, void *out, int64_t T, int64_t d, int64_t F,
                                int64_t L, int tying, int64_t t_begin, int64_t t_end, uint64_t src_mask, int dtype, int out_f32,
                                int64_t max_entries, void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype != CLT_BF16 && dtype != CLT_F16) return CLT_ERR_DTYPE;
  if (T < 0 || d <= 0 || F <= 0 || L <= 0 || L > 64 || d % SP_COLS != 0 || max_entries < 0) return CLT_ERR_ARG;
  if (t_begin < 0 || t_end > L || t_begin > t_end) return CLT_ERR_ARG;
  if (tying != CLT_TYING_NONE && tying != CLT_TYING_PER_SOURCE) return CLT_ERR_ARG;
  if (T == 0 || t_begin == t_end) return CLT_OK;
  if (!row_ptr || !col || !val || !w_packed || !out || !workspace) return CLT_ERR_ARG;
  if (!clt_aligned16(w_packed) || !clt_aligned16(out) || !clt_aligned16(workspace) || (bias_sum && !clt_aligned16(bias_sum)) ||
      (skip_add && !clt_aligned16(skip_add)))
    return CLT_ERR_ALIGN;
  const int64_t pitch = clt_pitch(d, 2);
  const SpLayout l = tile_layout(T, d, F, L, t_end - t_begin, max_entries);
  if (!sp_shape_ok(l, pitch * 2)) return CLT_ERR_RANGE;
  if (workspace_bytes < l.bytes) return CLT_ERR_WORKSPACE;
  RecArgs ra;
  ra.row_ptr = row_ptr; ra.col = col; ra.src = nullptr; ra.val = val; ra.Rn = T; ra.L = L; ra.max_entries = max_entries;
  ra.layer_mask = src_mask;
  sp_place_workspace(ra, l, (char *)workspace);
  TileArgs ta;
  ta.p = l.p; ta.counts = ra.counts; ta.total = ra.total; ta.recs = ra.recs;
  ta.wp = w_packed; ta.bias_sum = bias_sum; ta.skip_add = skip_add; ta.out = out;
  ta.row_ptr = row_ptr; ta.col = col; ta.val = val; ta.bad = ra.bad;
  ta.list_total = row_ptr + L * T; ta.max_entries = max_entries;
  ta.Tn = T; ta.d = d; ta.F = F; ta.L = L; ta.pitch = pitch; ta.src_mask = src_mask;
  ta.tying = tying; ta.t_begin = (int)t_begin; ta.t_end = (int)t_end; ta.out_f32 = out_f32; ta.col_parts = l.col_parts;
  if (dtype == CLT_BF16) return launch_tiles<bf16_t>(ra, ta, l.col_parts, (hipStream_t)stream);
  return launch_tiles<f16_t>(ra, ta, l.col_parts, (hipStream_t)stream);
}

extern "C" int clt_grad_tiles_supported(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries, int dtype) {
  if (dtype != CLT_BF16 || T <= 0 || d <= 0 || d % SP_COLS != 0 || F <= 0 || L <= 0 || L > 64 || entries < 0) return 0;
  const SpLayout l = grad_layout(T, d, F, L, entries);
  return sp_shape_ok(l, d * 2) && 8 * clt_ceil_div((int64_t)l.p.parts * l.col_parts, 8) * (L * (L + 1) / 2) <= 0x7FFFFFFFll;
}

extern "C" size_t clt_grad_tiles_workspace_bytes(int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries) {
  if (T <= 0 || d < SP_COLS || F <= 0 || L <= 0 || entries < 0) return 0;
  return grad_layout(T, d, F, L, entries).bytes;
}

static int grad_tiles(GradOut kind, const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val,
                      const void *g_model, float *out, void *const *params, int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries,
                      int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype != CLT_BF16) return CLT_ERR_DTYPE;
  if (!clt_grad_tiles_supported(T, d, F, L, entries, dtype)) return CLT_ERR_ARG;
  if (!list_ptr || !list_tok || !list_src || !val || !g_model || !(kind == GT_ROWS ? (const void *)out : (const void *)params) || !workspace)
    return CLT_ERR_ARG;
  if (!clt_aligned16(g_model) || !clt_aligned16(out) || !clt_aligned16(workspace)) return CLT_ERR_ALIGN;
  for (int64_t i = 0; kind == GT_PARAM && i < L * (L + 1) / 2; ++i) {
    if (!params[i]) return CLT_ERR_ARG;
    if (!clt_aligned16(params[i])) return CLT_ERR_ALIGN;
  }
  GradArgs a{};
  a.g = g_model; a.out = out;
  a.Tn = T; a.d = d; a.F = F; a.L = L; a.max_entries = entries;
  return launch_grad(kind, list_ptr, list_tok, list_src, val, a, params, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int clt_decoder_grad_tiles(const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val,
                                      const void *g_model, float *out, int64_t T, int64_t d, int64_t F, int64_t L, int64_t entries,
                                      int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  return grad_tiles(GT_ROWS, list_ptr, list_tok, list_src, val, g_model, out, nullptr, T, d, F, L, entries, dtype, workspace,
                    workspace_bytes, stream);
}

extern "C" int clt_decoder_grad_params_tiles(const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val,
                                             const void *g_model, void *const *outs, int64_t T, int64_t d, int64_t F, int64_t L,
                                             int64_t entries, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  if (F % 8 != 0) return CLT_ERR_ARG;
  return grad_tiles(GT_PARAM, list_ptr, list_tok, list_src, val, g_model, nullptr, outs, T, d, F, L, entries, dtype, workspace,
                    workspace_bytes, stream);
}

extern "C" int clt_decoder_grad_param_tiles(const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val,
                                            const void *g_model, void *out, int64_t T, int64_t d, int64_t F, int64_t L,
                                            int64_t entries, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  if (!out || L <= 0 || L > 64) return CLT_ERR_ARG;
  void *outs[64 * 65 / 2];
  for (int64_t i = 0; i < L * (L + 1) / 2; ++i) outs[i] = (char *)out + i * d * F * 2;
  return clt_decoder_grad_params_tiles(list_ptr, list_tok, list_src, val, g_model, outs, T, d, F, L, entries, dtype, workspace,
                                       workspace_bytes, stream);
}

extern "C" int clt_decoder_grad_adam_tiles(const int32_t *list_ptr, const int32_t *list_tok, const int32_t *list_src, const void *val,
                                           const void *g_model, void *w_packed, float *m, float *v, int moments_by_tile, int64_t T,
                                           int64_t d, int64_t F, int64_t L, int64_t entries, double lr, double beta1, double beta2,
                                           double eps, int64_t step, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype != CLT_BF16) return CLT_ERR_DTYPE;
  if (!clt_grad_tiles_supported(T, d, F, L, entries, dtype)) return CLT_ERR_ARG;
  if (step < 1 || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1)) return CLT_ERR_ARG;
  if (!list_ptr || !list_tok || !list_src || !val || !g_model || !w_packed || !m || !v || !workspace) return CLT_ERR_ARG;
  if (!clt_aligned16(g_model) || !clt_aligned16(w_packed) || !clt_aligned16(m) || !clt_aligned16(v) || !clt_aligned16(workspace))
    return CLT_ERR_ALIGN;
  GradArgs a{};
  a.g = g_model; a.w = w_packed; a.m = m; a.v = v;
  a.Tn = T; a.d = d; a.F = F; a.L = L; a.pitch = clt_pitch(d, 2); a.max_entries = entries;
  a.m_dec = F * d;
  a.m_row = moments_by_tile ? SP_COLS : d;
  a.m_cols = moments_by_tile ? F * SP_COLS : SP_COLS;
  a.adam = adam_coef(lr, beta1, beta2, eps, step);
  return launch_grad(GT_ADAM, list_ptr, list_tok, list_src, val, a, nullptr, workspace, workspace_bytes, (hipStream_t)stream);
}
