// float32 mode on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands and
// sums, no narrower type anywhere): the split-KV attention kernel for float32
// caches with kv_lora_rank 512 and qk_rope_head_dim 64, and the query
// absorption for float32 weights. The math is decode_generic_kernel's and
// absorb_kernel's (la_generic.hip), which keep the other shapes.
//
// decode_generic_kernel gives every query head its own workgroup, so 128 heads
// read every row 128 times through the L2 and reduce every score over a wave:
// 4 x 1000 rows and 128 heads took 377 us. Here a workgroup of 4 waves takes 16
// heads and walks tiles of 32 positions staged in LDS; two workgroups share a
// CU (76 KB each), one's loads under the other's matrix work.
// 4 x 1000 rows and 128 heads take 33 us (matrix cores 17.4K of 58.6K busy
// cycles; the rest is the latency of loads, barriers and softmax, which two
// workgroups only partly hide), 1 x 8192 37 us. Fewer heads than 16 multiply the
// 16-head tile all the same and gain as much (a whole step of one head, here and
// on decode_generic_kernel: 1 x 64 rows 26 / 152 us, 1 x 8192 30 / 415, 64 x 10
// 64 / 186).
//
// An MFMA step multiplies 4 k's, lane group g = lane / 16 holding one of them;
// which k's a step takes is free as long as both operands agree, so every
// operand is a 16-B load feeding four steps:
//   * scores: step (jj, e) takes k = 16 jj + 4 g + e; A = chunk 4 jj + g of the
//     tile row, B = the same elements of Q (in registers for the segment). Waves
//     split (position block of 16) x (half of the 576 elements); the halves
//     meet in LDS and every wave adds up all 32 x 16 scores, so the maximum, the
//     exponentials and their sum need no further exchange;
//   * PV: step (pb, i) takes positions 16 pb + 4 g + i, which is where the
//     score accumulators already hold them (B = P from registers); A = 4
//     consecutive latent columns of a value row, one per MFMA, so accumulator c
//     of a 64-column block holds its columns 4 m + c.
// Tile rows are unpadded; chunk j of row r sits at j ^ (r % 16): the score reads
// (16 rows at one chunk) and the value reads (16 chunks of a row) are
// conflict-free. The HBM->LDS copies write LDS linearly, so the permutation is
// applied to the global address each lane reads.
#include "la_internal.hpp"

namespace la {
namespace {

constexpr int kDc = 512;
constexpr int kDr = 64;
constexpr int kRowB = (kDc + kDr) * 4;
constexpr int kT = 32;  // positions per tile
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kCtPitch = kDc * 4;
constexpr int kRopeOff = kT * kCtPitch;          // 256-B k_rope rows
constexpr int kSumOff = kRopeOff + kT * kDr * 4;  // partial scores: [wave][lane] 16 B
constexpr int kLdsBytes = kSumOff + kWaves * 1024;
static_assert(2 * kLdsBytes <= 160 * 1024, "two workgroups per CU");

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) char lchar;

__device__ inline f32x4 lds_ld(const lchar* L, int off) {
  return *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(L + off);
}
__device__ inline void lds_st(lchar* L, int off, f32x4 v) {
  *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(L + off) = v;
}
__device__ inline f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <bool kPaged, bool kFilled>
__global__ __launch_bounds__(kThreads, 2) void decode_f32_kernel(DecodeProblem p, int groups, float* zero_out,
                                                                 int64_t zero_n) {
  warm_kernarg_lines(p);
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  lchar* L = (lchar*)lds_raw;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  // the output that a latent-half merge adds into: a grid-stride share each
  if (zero_out)
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < zero_n; i += (int64_t)gridDim.x * kThreads)
      zero_out[i] = 0.f;
  int chunk, group;
  block_coords(p.num_chunks, groups, &chunk, &group);
  if (chunk >= p.num_chunks) return;
  const int head0 = group * 16;

  ChunkWalk<kFilled> w;
  if (!walk_begin(p, chunk, group, w)) return;

  const int pb_w = wave & 1, kh = wave >> 1;  // this wave's score block and half of the row
  const int row_l = 16 * pb_w + n16;

  while (walk_next(p, w)) {
    const int s = w.s;
    const char* const seg_base = reinterpret_cast<const char*>(p.kv) + (kPaged ? 0 : (w.row0 + (w.lo - w.s_lo)) * kRowB);
    const uint32_t pos0 = (uint32_t)(w.lo - w.s_lo);
    const int last = (int)(w.seg_hi - w.lo - 1);
    const int ntiles = last / kT + 1;
    const int64_t rlim = p.rope_rows > 0 ? p.rope_rows - 1 : INT64_MAX;

    // Q[head0 + n16][16 jj + 4 g .. +3] of this wave's half (jj = 18 kh + i),
    // scaled; heads past the last one read it again (finite, never stored)
    f32x4 q[18];
    {
      const int64_t qrow = (int64_t)s * p.Hq + min(head0 + n16, p.Hq - 1);
#pragma unroll
      for (int i = 0; i < 18; ++i) {
        const int jj = 18 * kh + i;
        q[i] = *reinterpret_cast<const f32x4*>(jj < 32 ? p.q_abs + qrow * kDc + 16 * jj + 4 * g
                                                       : p.q_rope + qrow * kDr + 16 * (jj - 32) + 4 * g);
        q[i] *= p.scale_log2;
      }
    }
    f32x4 o[2][4];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int c = 0; c < 4; ++c) o[cb][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = 0; t < ntiles; ++t) {
      // ---- stage the wave's 8 rows (rows past the segment re-read its last) ----
      const int tb = min(kT * t + 8 * wave, last);  // first row; the 8 lie in one block of a paged cache
      const int left = last - tb;
      const char* base;
      if constexpr (kPaged) {
        const uint32_t pos = pos0 + (uint32_t)tb, tile = pos >> 5;
        const uint32_t blk = (__umulhi(tile, p.tpb_magic) + tile) >> p.tpb_shift;
        const int e = min(max(p.block_table[(int64_t)s * p.blocks_per_seq + blk], 0), p.pool_last);
        const uint32_t row = (uint32_t)e * (uint32_t)p.block_size + (pos - blk * (uint32_t)p.block_size);
        base = reinterpret_cast<const char*>(p.kv) + (uint64_t)row * kRowB;
      } else {
        base = seg_base + (int64_t)tb * kRowB;
      }
      // k_rope: lane takes row lane/8, pairs 4 (lane%8) .. +3
      const int rr = lane >> 3, u = lane & 7;
      const int rrow = min(rr, left);
      const int64_t rpos = min((int64_t)pos0 + tb + rrow, rlim);
      const f32x4* ks = reinterpret_cast<const f32x4*>(base + rrow * kRowB + kDc * 4);
      const f32x4 k0 = ks[u], k1 = ks[8 + u];
      const f32x4 cs = *reinterpret_cast<const f32x4*>(p.rope_cos + rpos * (kDr / 2) + 4 * u);
      const f32x4 sn = *reinterpret_cast<const f32x4*>(p.rope_sin + rpos * (kDr / 2) + 4 * u);
      if (t > 0) lds_barrier();  // every wave is done with the previous tile
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int f = (8 * wave + j) & 15;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __builtin_amdgcn_global_load_lds(base + (uint32_t)(min(j, left) * kRowB + 1024 * h + 16 * (lane ^ f)),
                                           (lds_void*)(L + (8 * wave + j) * kCtPitch + 1024 * h), 16, 0, 0);
      }
      {
        const int r = 8 * wave + rr;
        lds_st(L, kRopeOff + r * 256 + 16 * (u ^ (r & 15)), k0 * cs - k1 * sn);
        lds_st(L, kRopeOff + r * 256 + 16 * ((8 + u) ^ (r & 15)), k0 * sn + k1 * cs);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the copies have landed
      lds_barrier();
      // ---- partial scores of 16 positions over half of the row ----
      // k-half 0 is chunks 0 .. 71 of the c_t row, half 1 its chunks 72 .. 127
      // and the 16 of the k_rope row; row % 16 = n16
      // eight chains, added as a tree (one chain of 288 products was further
      // from 64 bits than the VALU kernel's sums)
      f32x4 sc[8] = {};
#pragma unroll
      for (int i = 0; i < 18; ++i) {
        const int jj = 18 * kh + i;  // wave-uniform
        const int off = jj < 32 ? row_l * kCtPitch + 16 * ((4 * jj + g) ^ n16)
                                : kRopeOff + row_l * 256 + 16 * ((4 * (jj - 32) + g) ^ n16);
        const f32x4 a = lds_ld(L, off);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f32x4& d = sc[4 * (i & 1) + e];
          d = mma(a[e], q[i][e], d);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) settle(sc[e]);
#pragma unroll
      for (int n = 4; n > 0; n >>= 1)
#pragma unroll
        for (int e = 0; e < n; ++e) sc[e] += sc[e + n];
      lds_st(L, kSumOff + 1024 * wave + 16 * lane, sc[0]);
      lds_barrier();
      // lane: head n16, positions 16 pb + 4 g + i
      f32x4 pr[2];
      const int valid = last + 1 - kT * t;
      float mx = m;
#pragma unroll
      for (int pb = 0; pb < 2; ++pb) {
        pr[pb] = lds_ld(L, kSumOff + 1024 * pb + 16 * lane) + lds_ld(L, kSumOff + 1024 * (pb + 2) + 16 * lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (16 * pb + 4 * g + i >= valid) pr[pb][i] = -INFINITY;
          mx = fmaxf(mx, pr[pb][i]);
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float alpha = exp2f(m - mx);
      const bool moved = mx != m;
      m = mx;
      float sum = 0.f;
#pragma unroll
      for (int pb = 0; pb < 2; ++pb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pr[pb][i] = exp2f(pr[pb][i] - m);
          sum += pr[pb][i];
        }
      l = l * alpha + sum;
      if (t > 0 && __builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
          for (int c = 0; c < 4; ++c) o[cb][c] *= alpha;
      }
      // ---- PV over this wave's 128 columns ----
#pragma unroll
      for (int pb = 0; pb < 2; ++pb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * pb + 4 * g + i;
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            const f32x4 a = lds_ld(L, r * kCtPitch + 16 * ((32 * wave + 16 * cb + n16) ^ (r & 15)));
#pragma unroll
            for (int c = 0; c < 4; ++c) o[cb][c] = mma(a[c], pr[pb][i], o[cb][c]);
          }
        }
    }

    // ---- segment end: O / l (fp32) and the base-2 log-sum-exp, as decode_generic_kernel writes them ----
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int c = 0; c < 4; ++c) settle(o[cb][c]);
    if (head0 + n16 < p.Hq) {
      const int64_t row = (kFilled ? slot_of(p, chunk, s) : (int64_t)chunk + s) * p.Hq + head0 + n16;
      const float inv = 1.f / l;
      // accumulator (cb, c), element r: column 128 wave + 64 cb + 4 (4 g + r) + c
      float* dst = p.part_o + row * kDc + 128 * wave + 16 * g;
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<f32x4*>(dst + 64 * cb + 4 * r) =
              f32x4{o[cb][0][r], o[cb][1][r], o[cb][2][r], o[cb][3][r]} * inv;
      if (wave == 0 && g == 0) p.part_lse[row] = m + log2f(l);
    }
    lds_barrier();  // the next segment's tile lands on this one's
    w.lo = w.seg_hi;
    ++w.s;
  }
}

// q_abs[t,h,c] = sum_i q_nope[t,h,i] W_UK[h dn + i, c], fp32. One wave per
// (head, 64 latent columns, 16 tokens): step (jj, e) takes i = 16 jj + 4 g + e,
// A = W's row i, 4 consecutive columns per lane (one per MFMA), B = q. W
// streams through registers once per 16 tokens (33.5 MB at 128 heads), eight
// 16-row groups of loads in flight per wave: 9.6 us for 4 tokens, where
// absorb_kernel (one column per thread, serial over i) took 52.8.
// kNJ = dn / 16 when known at compile time (8 for dn = 128), 0 for any multiple
// of 16.
constexpr int kAbsJ = 8;
template <int kNJ>
__global__ __launch_bounds__(256) void absorb_f32_kernel(const float* __restrict__ q_nope, const float* __restrict__ W,
                                                         float* __restrict__ q_abs, int tokens, int nh, int dn, int dc) {
  const int lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
  const int ncb = dc / 64;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);  // (head, 64-column block)
  const int h = item / ncb, c0 = 64 * (item - h * ncb);
  if (h >= nh) return;
  const int t = blockIdx.y * 16 + n16;
  const float* qr = q_nope + ((int64_t)min(t, tokens - 1) * nh + h) * dn + 4 * g;
  const float* wr = W + ((int64_t)h * dn + 4 * g) * dc + c0 + 4 * n16;
  f32x4 part[4][8] = {};  // eight chains per column, added as a tree
  const int nj = kNJ > 0 ? kNJ : dn / 16;
  for (int j0 = 0; j0 < nj; j0 += kAbsJ) {
    f32x4 w[kAbsJ][4], q[kAbsJ];
#pragma unroll
    for (int j = 0; j < kAbsJ; ++j) {
      const int jj = min(j0 + j, nj - 1);  // groups past the last are read again and not used
      q[j] = *reinterpret_cast<const f32x4*>(qr + 16 * jj);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[j][e] = *reinterpret_cast<const f32x4*>(wr + (int64_t)(16 * jj + e) * dc);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the group before its first use
#pragma unroll
    for (int j = 0; j < kAbsJ; ++j) {
      if (kNJ == 0 && j0 + j >= nj) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          f32x4& d = part[c][4 * (j & 1) + e];
          d = mma(w[j][e][c], q[j][e], d);
        }
    }
  }
  f32x4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int e = 0; e < 8; ++e) settle(part[c][e]);
#pragma unroll
    for (int n = 4; n > 0; n >>= 1)
#pragma unroll
      for (int e = 0; e < n; ++e) part[c][e] += part[c][e + n];
    acc[c] = part[c][0];
  }
  if (t >= tokens) return;
  // accumulator c, element r: column c0 + 4 (4 g + r) + c of token t
  float* dst = q_abs + ((int64_t)t * nh + h) * dc + c0 + 16 * g;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    *reinterpret_cast<f32x4*>(dst + 4 * r) = f32x4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
}

template <bool kPaged, bool kFilled>
hipError_t launch_f32_t(const DecodeProblem& p, hipStream_t stream, float* zero_out, int64_t zero_n) {
  static OncePerDevice once;
  const hipError_t e = allow_lds(once, reinterpret_cast<const void*>(&decode_f32_kernel<kPaged, kFilled>), kLdsBytes);
  if (e != hipSuccess) return e;
  const int groups = (p.Hq + 15) / 16;
  hipLaunchKernelGGL((decode_f32_kernel<kPaged, kFilled>), dim3((unsigned)mfma_grid_blocks(p.num_chunks, groups)), dim3(kThreads),
                     kLdsBytes, stream, p, groups, zero_out, zero_n);
  return hipGetLastError();
}

}  // namespace

bool decode_f32_supported(const DecodeProblem& p) {
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return p.kv_dtype == LA_DTYPE_F32 && p.dc == kDc && p.dR == kDr && aligned(p.kv) && aligned(p.q_abs) &&
         aligned(p.q_rope) && aligned(p.rope_cos) && aligned(p.rope_sin) &&
         // 32-bit sequence lookup and positions (find_seq_mfma); tiles inside one block of a paged cache
         (p.offsets || (int64_t)p.num_seqs * p.seq_len <= INT32_MAX) && p.total_rows <= INT32_MAX &&
         (!p.block_table || p.block_size % kT == 0) && device_is_gfx950();
}

hipError_t launch_decode_f32(const DecodeProblem& p, hipStream_t stream, float* zero_out, int64_t zero_n) {
  if (p.block_table) return launch_f32_t<true, true>(p, stream, zero_out, zero_n);
  return p.chunk_len < 0 ? launch_f32_t<false, true>(p, stream, zero_out, zero_n)
                         : launch_f32_t<false, false>(p, stream, zero_out, zero_n);
}

bool absorb_f32_supported(const void* q_nope, const void* W, int w_dtype, const float* q_abs, int dn, int dc) {
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return w_dtype == LA_DTYPE_F32 && dn % 16 == 0 && dc % 64 == 0 && aligned(q_nope) && aligned(W) && aligned(q_abs) &&
         device_is_gfx950();
}

hipError_t launch_absorb_f32(const float* q_nope, const void* W, float* q_abs, int tokens, int nh, int dn, int dc,
                             hipStream_t stream) {
  const dim3 grid((unsigned)((nh * (dc / 64) + 3) / 4), (unsigned)((tokens + 15) / 16));
  auto k = dn == 128 ? absorb_f32_kernel<8> : absorb_f32_kernel<0>;
  hipLaunchKernelGGL(k, grid, dim3(256), 0, stream, q_nope, reinterpret_cast<const float*>(W), q_abs,
                     tokens, nh, dn, dc);
  return hipGetLastError();
}

}  // namespace la
