// Internal types shared by the HIP kernels and the C-ABI layer of
// liblatent_attn_hip.so. Not installed; the public ABI is include/latent_attn.h.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <cstddef>
#include <cstdint>

#include "la_once.hpp"
#include "latent_attn.h"

namespace la {

// log2(e): scores are kept in base-2 units so the softmax uses v_exp_f32 (2^x).
constexpr float kLog2e = 1.4426950408889634f;

// One decode step, fully resolved on the host. Passed to kernels by value.
//
// Sequences: sequence s owns rows [seq_begin(s), seq_begin(s+1)) of the packed
// cache; RoPE positions are row - seq_begin(s). Each sequence carries Hq query
// heads = queries_per_seq * nh; query row (s, hq) reads q_abs[(s*Hq + hq)*dc].
//
// Split-KV plan: the flat row space is cut into num_chunks chunks of
// chunk_len rows. The piece of chunk c that falls in sequence s is one
// "segment"; it writes partial slot (c + s): part_o[(slot*Hq + hq)*dc + i]
// (normalised by its own softmax sum) and part_lse[slot*Hq + hq] (base-2
// log-sum-exp of the scaled scores). Slots are unique because a sequence's
// chunks form a contiguous range that starts no earlier than where the
// previous sequence's range ends; num_slots = num_chunks + num_seqs - 1.
// q_prep layout of the MFMA path ("operand order"). The query rows of each
// sequence are padded to a multiple of 32 (qprep_rows_per_seq) and cut into
// blocks of 32 rows (qrow = s * qprep_rows_per_seq(Hq) + hq). Block b stores,
// for k-step kk (16 elements of the 576-element row) and lane l = r + 32 g,
// the 8 elements Q[32 b + r][16 kk + 8 g .. +8] at element 512 kk + 8 l: the
// attention kernel's B operand of k-step kk is one coalesced 1 KB load.
constexpr int kQPrepRow = 576;  // kv_lora_rank 512 + qk_rope_head_dim 64
__host__ __device__ inline int qprep_rows_per_seq(int Hq) { return (Hq + 31) & ~31; }
__host__ __device__ inline int64_t qprep_index(int64_t qrow, int c) {
  return (qrow >> 5) * (32 * kQPrepRow) + 512 * (c >> 4) + 8 * ((qrow & 31) + 32 * ((c >> 3) & 1)) + (c & 7);
}

// Longest chunk, or piece of filled rows, that the MFMA kernels take: keeps row byte offsets inside 32 bits.
constexpr int kMaxChunkRows = 1 << 20;

struct DecodeProblem {
  const void* kv;
  int kv_dtype;
  int row_elems;  // dc + dR
  int64_t total_rows;
  int num_seqs;
  int seq_len;            // used when offsets == nullptr
  const int32_t* offsets; // device, num_seqs + 1, or nullptr
  const int32_t* lens;    // device, num_seqs, or nullptr: filled rows of each region
  // paged cache (block_table != nullptr): kv is a pool of pool_blocks blocks
  // of block_size rows; the row space above is virtual (sequence s owns
  // [s * seq_len, (s+1) * seq_len), seq_len = blocks_per_seq * block_size),
  // position pos of sequence s lives in pool row paged_row(p, s, pos)
  const int32_t* block_table;  // device, num_seqs * blocks_per_seq
  int block_size;
  int blocks_per_seq;
  int64_t pool_blocks;
  // paged MFMA kernel (block_size % 32 == 0): 32-row tiles per block and the
  // multiplier that divides by it, q / tile_per_block = (mulhi(q, tpb_magic)
  // + q) >> tpb_shift for q < 2^31 (set by set_tile_divisor); pool_last =
  // pool_blocks - 1, capped at INT32_MAX (table entries are int32)
  uint32_t tile_per_block, tpb_magic;
  int tpb_shift;
  int pool_last;
  int qps;                // query tokens per sequence
  int nh;                 // weight heads
  int Hq;                 // query heads per sequence = qps * nh
  int merge_rows_log2;    // half-row merge: log2 of its query rows per workgroup (in the padding before
                          // the pointers, which one load brings with the three above)
  const float* q_abs;     // (num_seqs*Hq, dc) f32
  const float* q_rope;    // (num_seqs*Hq, dR) f32
  void* q_prep;           // MFMA path: [q_abs | q_rope] * scale_log2 in the MFMAs' 16-bit
                          // type, operand-order layout (qprep_index), written by
                          // launch_prep_q or the absorb kernel
  const void* W_UV;
  int wuv_dtype;
  const float* rope_cos;
  const float* rope_sin;
  int64_t rope_rows;      // 0 = unchecked
  float* out;             // (num_seqs*Hq, dv)
  int dc, dR, dv;
  float scale_log2;       // softmax scale * log2(e)
  // plan
  int chunk_len;       // rows per chunk, or < 0: the filled rows divided on the device (below)
  int num_chunks;
  int num_slots;
  float* part_o;       // fp32 rows O / l, or (part_f16) fp16 rows, see below
  float* part_lse;     // base-2 log-sum-exp m + log2(l) of the slot's scores
  // part_f16 (MFMA kernel): part_o row (slot, hq) holds the unnormalised
  // numerator N = sum_pos 2^(s_pos - m) V_pos as fp16 N * 2^-e, with e chosen
  // per half row (columns 0..255, 256..511) so every value is below 1;
  // part_scale[2 row + half] = 2^e and part_m[row] = m. O / l = N / l with
  // 1 / l = 2^(m - lse).
  int part_f16;
  float* part_scale;
  float* part_m;
};

// One scalar load from each 64-B scalar-cache line of a DecodeProblem kernel
// argument (fields at 0x1c, 0x60, 0xa0 and 0xc4 of the 248-B struct; the
// int after it shares the last line), issued together at kernel start. The
// compiler loads every other field where it is first used, after branches on
// earlier ones; at kernel start the lines are cold, so each such round costs
// a full memory round trip (about 700 cycles), and the attention kernel's
// prologue took six of them before its first copy went out. With the lines
// warmed in one round, those loads hit the scalar cache.
__device__ inline void warm_kernarg_lines(const DecodeProblem& p) {
  asm volatile("" ::"s"(p.seq_len), "s"(p.Hq), "s"(p.rope_rows), "s"(p.num_chunks));
}
static_assert(offsetof(DecodeProblem, merge_rows_log2) == offsetof(DecodeProblem, qps) + 12, "one 16-B load");
static_assert(offsetof(DecodeProblem, seq_len) < 64 && offsetof(DecodeProblem, Hq) / 64 == 1 &&
                  offsetof(DecodeProblem, rope_rows) / 64 == 2 && offsetof(DecodeProblem, num_chunks) / 64 == 3 &&
                  sizeof(DecodeProblem) + 4 <= 256,
              "warm_kernarg_lines touches every 64-B line of the arguments");

// Partial row (slot, hq) element i as fp32 O / l.
__device__ inline float load_part(const DecodeProblem& p, int64_t row, int i) {
  if (p.part_f16)
    return (float)reinterpret_cast<const _Float16*>(p.part_o)[row * p.dc + i] * p.part_scale[2 * row + (i >= 256)] *
           exp2f(p.part_m[row] - p.part_lse[row]);
  return p.part_o[row * p.dc + i];
}

// First row of sequence s, clamped into [0, total_rows] so that malformed
// offsets can give wrong answers but never out-of-bounds reads.
__device__ inline int64_t seq_begin(const DecodeProblem& p, int s) {
  const int64_t b = p.offsets ? (int64_t)p.offsets[s] : (int64_t)s * p.seq_len;
  return b < 0 ? 0 : (b > p.total_rows ? p.total_rows : b);
}

// End of sequence s's rows: the end of its region, or, with per-sequence
// lengths, its first row plus its length clamped into the region (the rows
// past it are unfilled capacity and belong to no sequence).
__device__ inline int64_t seq_end(const DecodeProblem& p, int s) {
  const int64_t region_end = seq_begin(p, s + 1);
  if (!p.lens) return region_end;
  const int64_t b = seq_begin(p, s);
  const int64_t l = p.lens[s];
  return l <= 0 ? b : (b + l < region_end ? b + l : region_end);
}

// Division by an invariant d >= 1 with a multiply (Granlund & Montgomery,
// "Division by invariant integers using multiplication", PLDI 1994, the
// round-up multiplier): l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1,
// then q / d = (floor(q m / 2^32) + q) >> l for every q < 2^31 (the sum fits
// in 32 bits there).
inline void set_tile_divisor(DecodeProblem& p, uint32_t d) {
  int l = 0;
  while ((1ull << l) < d) ++l;
  p.tile_per_block = d;
  p.tpb_shift = l;
  p.tpb_magic = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
}

// Pool row of position pos of sequence s in a paged cache. Block ids are
// clamped into the pool: a malformed table gives wrong rows, never an
// out-of-bounds access. Requires pos < blocks_per_seq * block_size.
__device__ inline int64_t paged_row(const DecodeProblem& p, int s, int64_t pos) {
  int64_t b = p.block_table[(int64_t)s * p.blocks_per_seq + pos / p.block_size];
  b = b < 0 ? 0 : (b >= p.pool_blocks ? p.pool_blocks - 1 : b);
  return b * p.block_size + pos % p.block_size;
}

// RoPE table row of in-sequence position pos.
__device__ inline int64_t rope_row(const DecodeProblem& p, int64_t pos) {
  return (p.rope_rows > 0 && pos >= p.rope_rows) ? p.rope_rows - 1 : pos;
}

// Sequence whose row range contains row r: the largest s with
// seq_begin(s) <= r (empty sequences are skipped because their successor has
// the same begin). Requires seq_begin(0) <= r < seq_begin(num_seqs).
__device__ inline int find_seq(const DecodeProblem& p, int64_t r) {
  if (!p.offsets) return (int)(r / p.seq_len);
  int lo = 0, hi = p.num_seqs - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if ((int64_t)p.offsets[mid] <= r) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Block id -> (chunk, head group), XCD-aware. Workgroups are dispatched
// round-robin over the 8 XCDs (id % 8), each with its own L2. The work items
// (chunk, group), chunk-major, are cut into 8 contiguous ranges, one per XCD
// (XCD x: items [x*per, (x+1)*per), id = 8 k + x is item x*per + k). With
// one head group per chunk the chunks of one sequence share an L2, so the
// sequence's Q rows are fetched from HBM once per XCD rather than once per
// chunk, and every XCD streams one contiguous piece of the cache; with many
// head groups (several queries over one cache) the groups of a chunk share an
// L2 and its rows, and every XCD has work even when there are fewer chunks
// than XCDs. Ids past the last item return at once (chunk >= num_chunks).
__host__ __device__ inline int64_t mfma_grid_blocks(int num_chunks, int groups) {
  return 8 * (((int64_t)num_chunks * groups + 7) / 8);
}
// 32-bit arithmetic: the grid (8 per blocks) is below 2^31, so every item
// is (a 64-bit division here is ~130 dependent scalar instructions at the
// kernel's start).
__device__ inline void block_coords(int num_chunks, int groups, int* chunk, int* group) {
  const uint32_t id = blockIdx.x;
  const uint32_t per = ((uint32_t)num_chunks * (uint32_t)groups + 7) / 8;
  const uint32_t item = (id & 7) * per + (id >> 3);
  if (groups == 1) {
    *group = 0;
    *chunk = (int)item;
  } else {
    const uint32_t c = item / (uint32_t)groups;
    *group = (int)(item - c * (uint32_t)groups);
    *chunk = (int)c;
  }
}

// find_seq for the MFMA kernels: with uniform sequences the row space is
// below 2^31 rows (mfma_supported), so the division is a 32-bit one.
__device__ inline int find_seq_mfma(const DecodeProblem& p, int64_t r) {
  if (p.offsets) return find_seq(p, r);
  return (int)((uint32_t)r / (uint32_t)p.seq_len);
}

// Chunks over filled rows (chunk_len < 0; MFMA attention kernels with
// per-sequence lengths and no chunk_rows override). Regions are capacity: cut
// like the other plans' row space, the chunks over unfilled rows leave their
// workgroups idle and the others with a longer piece each (16 sequences of 300
// to 6000 rows in 6016-row regions, FP8, 128 heads: attention
// 36.4 us against 29.7).
// Instead every sequence is cut into pieces of its own of at most L rows, and
// piece c (counted over the sequences) is chunk c of a row space in which each
// sequence is padded to a multiple of L (filled_piece: at most num_chunks
// pieces), and no workgroup has a second segment (pieces across sequences, at
// their mean length, made the step 8 us slower: a segment's fixed part is that
// of eight tiles). The lengths are on the device, so every wave of the
// attention kernel sums them itself (wave-uniform code, all lanes active), and
// its workgroups leave what the merge needs in free slots
// (filled_notes): summed again there, behind its weight loads, it cost 1.5 us.
// The lane index is made in a volatile asm statement at each use, so that what
// derives from it is not held across loops, beside the operands in registers.
__device__ inline int wave_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}
// Inclusive sum over the lanes (DPP row shifts and broadcasts: no lane index).
__device__ inline int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ inline int wave_sum_i(int v) { return __builtin_amdgcn_readlane(wave_scan(v), 63); }
__device__ inline int filled_rows(const DecodeProblem& p, int s) {
  return (int)max(seq_end(p, s) - seq_begin(p, s), (int64_t)0);
}
__device__ inline int pieces(int rows, int len) { return (int)(((uint32_t)rows + (uint32_t)len - 1) / (uint32_t)len); }
// Rows of a piece when n pieces share total rows, at least the plan's shortest. The plan cuts filled rows only
// where the longest piece of its whole row space is a length that the kernels take.
__host__ __device__ inline int piece_rows(uint32_t total, uint32_t n, int shortest) {
  const int rows = (int)(((total + n - 1) / n + 31) & ~31u);
  return rows > shortest ? rows : shortest;
}
// Piece c: its sequence (num_seqs if there is none), that sequence's rows and
// first piece, and L, the fewest rows (a multiple of 32, at least -chunk_len)
// that num_chunks pieces suffice for: T / num_chunks at best,
// T / (num_chunks - num_seqs) always. The first 64 lengths stay in registers.
struct FilledPiece {
  int s, rows, first, len;
};
__device__ inline FilledPiece filled_piece(const DecodeProblem& p, int c) {
  const int lane = wave_lane();
  const int mine = lane < p.num_seqs ? filled_rows(p, lane) : 0;
  int t = mine;
  for (int i = lane + 64; i < p.num_seqs; i += 64) t += filled_rows(p, i);
  const uint32_t total = (uint32_t)wave_sum_i(t);
  // (malformed offsets can add up to more than the row space: their pieces stay within the kernels' length)
  auto share = [&](uint32_t n) { return min(piece_rows(total, n, -p.chunk_len), kMaxChunkRows); };
  auto fits = [&](int len) {
    int n = pieces(mine, len);
    for (int i = lane + 64; i < p.num_seqs; i += 64) n += pieces(filled_rows(p, i), len);
    return wave_sum_i(n) <= p.num_chunks;
  };
  int lo = share((uint32_t)p.num_chunks), hi = share((uint32_t)(p.num_chunks - p.num_seqs));
  if (lo != hi && fits(lo)) hi = lo;  // equal sequences take one try
  else lo = min(lo + 32, hi);
  while (lo < hi) {
    const int mid = (lo + hi) / 2 & ~31;  // lo <= mid < hi
    if (fits(mid)) hi = mid;
    else lo = mid + 32;
  }
  FilledPiece f{p.num_seqs, 0, 0, hi};
  for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
    const int rows = s0 == 0 ? mine : s0 + lane < p.num_seqs ? filled_rows(p, s0 + lane) : 0;
    const int n = pieces(rows, hi), end = wave_scan(n);
    const uint64_t past = __builtin_amdgcn_ballot_w64(f.first + end > c);
    if (past) {
      const int k = __builtin_ctzll(past);
      f.s = s0 + k;
      f.rows = __builtin_amdgcn_readlane(rows, k);
      f.first += __builtin_amdgcn_readlane(end, k) - __builtin_amdgcn_readlane(n, k);
      break;
    }
    f.first += __builtin_amdgcn_readlane(end, 63);
  }
  return f;
}
// First chunk of every sequence with rows, then L, written by the attention
// kernel's first workgroup of each sequence and of the launch. A piece lies in
// one sequence, so chunk c writes slot c and the num_seqs - 1 slots after the
// chunks' are free: the notes (num_seqs + 1 words) take their partial rows (at
// least 1 KB each), and the workspace is that of the other plans. One sequence
// has no free slot and needs no notes: seq_in_plan divides its rows itself.
__device__ inline int32_t* filled_notes(const DecodeProblem& p) {
  return reinterpret_cast<int32_t*>(reinterpret_cast<char*>(p.part_o) +
                                    (int64_t)p.num_chunks * p.Hq * p.dc * (p.part_f16 ? 2 : 4));
}
// Partial slot of the piece of chunk c inside sequence s.
__device__ inline int64_t slot_of(const DecodeProblem& p, int64_t c, int s) { return c + (p.chunk_len < 0 ? 0 : s); }
// A walk over the segments of one chunk (pieces of it inside one sequence).
// kFilled: 0, chunks of the regions only (such a kernel keeps the other code,
// and the registers it holds for later segments, out of its way to the first
// copy); 1, chunk_len may be < 0; 2, it is (one segment: with the code of the
// others beside it the 128-head kernel's body spilled two registers).
template <int kFilled>
struct ChunkWalk {
  int64_t lo, hi;  // what is left of the chunk, in the plan's row space
  int s;           // sequence of the current segment
  int64_t row0;    // first row of that sequence in the cache (its region)
  int64_t s_lo;    // and in the plan's row space
  int64_t seg_hi;  // end of the current segment there
};
template <int kFilled>
__device__ inline bool walk_begin(const DecodeProblem& p, int chunk, int group, ChunkWalk<kFilled>& w) {
  if (kFilled == 2 || (kFilled && p.chunk_len < 0)) {
    const FilledPiece f = filled_piece(p, chunk);
    // the last two: malformed offsets, whose sums wrap
    if (f.s >= p.num_seqs || chunk < f.first || (int64_t)(chunk - f.first) * f.len >= f.rows) return false;
    w.s = f.s;
    w.s_lo = (int64_t)f.first * f.len;
    w.row0 = seq_begin(p, f.s);
    w.lo = (int64_t)chunk * f.len;
    w.hi = w.seg_hi = min(w.lo + f.len, w.s_lo + f.rows);
    if (p.num_seqs > 1 && group == 0) {  // the same from every lane
      if (chunk == f.first) filled_notes(p)[f.s] = f.first;
      if (chunk == 0) filled_notes(p)[p.num_seqs] = f.len;
    }
    return true;
  }
  const int64_t end_all = seq_begin(p, p.num_seqs);
  w.lo = (int64_t)chunk * p.chunk_len;
  w.hi = min(w.lo + (int64_t)p.chunk_len, end_all);
  w.lo = max(w.lo, seq_begin(p, 0));
  if (w.lo >= w.hi) return false;
  w.s = find_seq_mfma(p, w.lo);
  return true;
}
// The next segment [lo, seg_hi) of sequence s; after it the caller sets lo = seg_hi and ++s.
template <int kFilled>
__device__ inline bool walk_next(const DecodeProblem& p, ChunkWalk<kFilled>& w) {
  while (w.lo < w.hi) {
    if (kFilled == 2 || (kFilled && p.chunk_len < 0)) return true;  // the one segment, set by walk_begin
    w.s_lo = w.row0 = seq_begin(p, w.s);
    w.lo = max(w.lo, w.s_lo);  // past the unfilled rows of the previous region
    if (w.lo >= w.hi) return false;
    const int64_t s_hi = seq_end(p, w.s);
    if (s_hi <= w.lo) {  // empty sequence, or lo in its unfilled rows
      if (++w.s >= p.num_seqs) return false;
      continue;
    }
    w.seg_hi = min(w.hi, s_hi);
    return true;
  }
  return false;
}

// Rows [lo, hi) of sequence s in the plan's row space, and the rows per chunk.
__device__ inline int seq_in_plan(const DecodeProblem& p, int s, int64_t* lo, int64_t* hi) {
  if (p.chunk_len < 0) {
    *hi = *lo = 0;
    const int rows = filled_rows(p, s);
    if (rows == 0) return 1;
    if (p.num_seqs == 1) {  // as filled_piece: num_chunks pieces always suffice
      *hi = rows;
      return piece_rows((uint32_t)rows, (uint32_t)p.num_chunks, -p.chunk_len);
    }
    // clamped into the plan: malformed offsets can leave notes unwritten (their
    // row sum wraps), which gives wrong answers but no access out of bounds
    const int len = max(filled_notes(p)[p.num_seqs], 1);
    *lo = (int64_t)min(max(filled_notes(p)[s], 0), p.num_chunks - 1) * len;
    *hi = min(*lo + rows, (int64_t)p.num_chunks * len);
    return len;
  }
  *lo = seq_begin(p, s);
  *hi = seq_end(p, s);
  return p.chunk_len;
}

// OCP FP8 E4M3 (e4m3fn) latent-cache element: sign, 4 exponent bits (bias
// 7), 3 mantissa bits; exponent 0 is subnormal (m * 2^-9), 0x7F / 0xFF NaN.
struct fp8e4m3 {
  uint8_t bits;
};
__device__ inline float fp8_to_f32(uint32_t c) {
  const uint32_t e = (c >> 3) & 15, m = c & 7;
  float v;
  if (e == 15 && m == 7) v = __builtin_nanf("");
  else if (e == 0) v = (float)m * 0x1p-9f;
  else v = __builtin_amdgcn_ldexpf(1.f + (float)m * 0.125f, (int)e - 7);
  return (c & 0x80) ? -v : v;
}
// Round to nearest even, saturating at +-448 (the largest finite value);
// NaN stays NaN.
__device__ inline uint8_t f32_to_fp8(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const uint32_t s = (b >> 24) & 0x80;
  const float a = __builtin_fabsf(x);
  if (a != a) return (uint8_t)(s | 0x7F);
  if (a >= 448.f) return (uint8_t)(s | 0x7E);
  if (a < 0x1p-6f) return (uint8_t)(s | (uint32_t)__builtin_rintf(a * 512.f));  // subnormal; 8 = 2^-6
  const uint32_t ab = __builtin_bit_cast(uint32_t, a);
  uint32_t e = ((ab >> 23) & 0xFF) - 127 + 7;  // 1 .. 15
  uint32_t m = (ab >> 20) & 7;
  const uint32_t rem = ab & 0xFFFFF;
  if (rem > 0x80000 || (rem == 0x80000 && (m & 1))) ++m;
  if (m == 8) {
    m = 0;
    ++e;
  }
  const uint32_t c = (e << 3) | m;
  return (uint8_t)(s | (c > 0x7E ? 0x7E : c));
}

template <typename T>
__device__ inline float to_f32(T v);
template <>
__device__ inline float to_f32<float>(float v) { return v; }
template <>
__device__ inline float to_f32<__half>(__half v) { return __half2float(v); }
template <>
__device__ inline float to_f32<__hip_bfloat16>(__hip_bfloat16 v) { return __bfloat162float(v); }
template <>
__device__ inline float to_f32<fp8e4m3>(fp8e4m3 v) { return fp8_to_f32(v.bits); }

// Load element i of a weight matrix whose dtype is only known at run time
// (uniform across the launch, so the switch does not diverge).
__device__ inline float load_any(const void* base, int dtype, int64_t i) {
  if (dtype == LA_DTYPE_BF16) return __bfloat162float(reinterpret_cast<const __hip_bfloat16*>(base)[i]);
  if (dtype == LA_DTYPE_F16) return __half2float(reinterpret_cast<const __half*>(base)[i]);
  if (dtype == LA_DTYPE_FP8_E4M3) return fp8_to_f32(reinterpret_cast<const uint8_t*>(base)[i]);
  return reinterpret_cast<const float*>(base)[i];
}

// LDS-visibility barrier that leaves outstanding HBM->LDS copies in flight.
// The "memory" clobber keeps the compiler from moving LDS accesses across it.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// 16 wait states between the last MFMA writing d and its first VALU reader (the
// compiler adds none where a branch lies between the two: row maxima were taken
// of unfinished scores).
template <typename V>
__device__ inline void settle(V& d) { asm volatile("s_nop 15" : "+v"(d)); }

__device__ inline float f_of(unsigned u) { return __builtin_bit_cast(float, u); }
__device__ inline unsigned u_of(float f) { return __builtin_bit_cast(unsigned, f); }
// x[l] + x[l ^ 32]
__device__ inline float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(u_of(x), u_of(x), false, false);
  return f_of(r[0]) + f_of(r[1]);
}

__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ inline float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// One la_append_kv call, resolved on the host (la_append.hip).
struct AppendProblem {
  void* kv;
  int kv_dtype;
  int64_t total_rows;
  int num_seqs;
  int capacity;            // region rows per sequence when offsets == nullptr
  const int32_t* offsets;  // device, num_seqs + 1, or nullptr
  int32_t* lens;           // device, num_seqs
  int tokens;
  const void* c_t;
  const void* k_rope;
  int src_dtype;
  float* q_rope;           // nullptr = no query rotation
  int qps;
  int nh;
  const float* rope_cos;
  const float* rope_sin;
  int64_t rope_rows;
  int32_t* status;
  int dc, dR;
  // paged cache (block_table != nullptr): as in DecodeProblem; capacity =
  // blocks_per_seq * block_size, kv a pool of pool_blocks blocks
  const int32_t* block_table;
  int block_size;
  int blocks_per_seq;
  int64_t pool_blocks;
};

// One la_naive_mla call (la_naive.hip): a single query over one cache.
struct NaiveProblem {
  const void* kv;
  int kv_dtype;
  int S;
  const void* W_UK;
  int wuk_dtype;
  const void* W_UV;
  int wuv_dtype;
  const float* q_nope;
  const float* q_rope;
  const float* rope_cos;
  const float* rope_sin;
  int64_t rope_rows;
  float* out;
  int nh, dn, dR, dc, dv;
  float scale;
  float* Kn;      // workspace: (S, nh*dn) fp32
  float* V;       // workspace: (S, nh*dv) fp32
  float* scores;  // workspace: (nh, S) fp32
};

// ---- host launchers (one per kernel family) -------------------------------

// Decompress-then-attend (la_naive.hip).
size_t naive_workspace_bytes(int64_t S, int nh, int dn, int dv);
hipError_t launch_naive(NaiveProblem p, void* workspace, hipStream_t stream);

// Device-side cache append + query RoPE.
hipError_t launch_append(const AppendProblem& p, hipStream_t stream);

// VALU split-KV decode: any dtype, kv_lora_rank <= 1024, qk_rope_head_dim <= 256.
hipError_t launch_decode_generic(const DecodeProblem& p, hipStream_t stream);
bool generic_supported(const DecodeProblem& p);

// Raises a kernel's dynamic LDS limit on the current device; each kernel has an OncePerDevice of its own.
inline hipError_t allow_lds(OncePerDevice& once, const void* fn, int bytes) {
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  return once.run(dev, [&] { return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes); });
}

// Whether the current device runs the MFMA kernels.
bool device_is_gfx950();

// fp32 split-KV decode and absorption on the fp32 MFMA (la_f32.hip): float32
// caches with kv_lora_rank 512, qk_rope_head_dim 64; float32 weights. zero_out
// (optional): zero_n floats the attention kernel zeroes for a half-row merge.
bool decode_f32_supported(const DecodeProblem& p);
hipError_t launch_decode_f32(const DecodeProblem& p, hipStream_t stream, float* zero_out = nullptr, int64_t zero_n = 0);
bool absorb_f32_supported(const void* q_nope, const void* W_UK, int w_dtype, const float* q_abs, int dn, int dc);
hipError_t launch_absorb_f32(const float* q_nope, const void* W_UK, float* q_abs, int tokens, int nh, int dn, int dc,
                             hipStream_t stream);

// MFMA split-KV decode for 16-bit and FP8 E4M3 caches with kv_lora_rank 512,
// qk_rope_head_dim 64.
// ev_begin / ev_end (optional) are recorded at the kernel's start and end.
hipError_t launch_decode_mfma(const DecodeProblem& p, hipStream_t stream, hipEvent_t ev_begin = nullptr,
                              hipEvent_t ev_end = nullptr);
bool mfma_supported(const DecodeProblem& p);
// The same with 16 query heads per workgroup (la_mfma16.hip); waves = 4 or 8
// per workgroup (tiles of 64 or 128 positions).
// With 8 waves and no q_prep it takes the fp32 queries; zero_out (optional): zero_n floats
// it zeroes for a latent-half merge.
hipError_t launch_decode_mfma16(const DecodeProblem& p, int waves, hipStream_t stream, float* zero_out, int64_t zero_n,
                                hipEvent_t ev_begin = nullptr, hipEvent_t ev_end = nullptr);
// The attention kernel's grid and copy schedule with no compute (a
// streaming-ceiling measurement); ring = 3 or 4 tile buffers. 16-bit
// contiguous caches.
hipError_t launch_stream_copies(const DecodeProblem& p, int ring, hipStream_t stream);
int mfma_heads_per_group();
// Fills p.q_prep from p.q_abs and p.q_rope (MFMA path only).
// zero_out (optional): zero_n floats zeroed for a latent-half merge.
hipError_t launch_prep_q(const DecodeProblem& p, hipStream_t stream, float* zero_out = nullptr, int64_t zero_n = 0);

// log-sum-exp combine of the partial slots + W_UV projection into p.out.
hipError_t launch_combine_project(const DecodeProblem& p, hipStream_t stream);

// MFMA versions for 16-bit weights (la_proj.hip).
bool absorb_mfma_supported(int w_dtype, int nh, int dn, int dc);
// out_mode 0: out = q_abs (fp32). 1 / 2: out = q_prep (bf16 / fp16) =
// [q_abs | q_rope] * scale in the operand-order layout, as prep_q_kernel
// writes it; token t is query t % qps of sequence t / qps (qps = tokens per
// sequence, used by modes 1 / 2 only).
// zero_out (optional): zero_n floats the kernel zeroes, for a merge that adds
// its latent halves into the output.
hipError_t launch_absorb_mfma(const float* q_nope, const void* W_UK, int w_dtype, void* out, int out_mode,
                              const float* q_rope, float scale, int dR, int tokens, int nh, int dn, int dc, int qps,
                              hipStream_t stream, float* zero_out = nullptr, int64_t zero_n = 0);
bool project_mfma_supported(const DecodeProblem& p);
// Workgroups of the full-row merge + projection launch.
int merge_project_blocks(const DecodeProblem& p);
// Merge of the split partials and W_UV projection in one kernel (the merged
// rows stay in LDS: no workspace). halves: one workgroup per latent half,
// which adds its product into p.out with atomics: p.out must be zero (fp16
// partials only). ncu: the device's compute units.
hipError_t launch_combine_project_mfma(const DecodeProblem& p, hipStream_t stream, bool halves, int ncu);

// The same in fp32 for float32 weights; halves as above (any partial format).
bool project_f32_supported(const DecodeProblem& p);
hipError_t launch_combine_project_f32(const DecodeProblem& p, hipStream_t stream, bool halves);

// q_abs = q_nope . W_UK per head.
hipError_t launch_absorb(const float* q_nope, const void* W_UK, int w_dtype, float* q_abs, int tokens, int nh, int dn,
                         int dc, hipStream_t stream);

}  // namespace la
