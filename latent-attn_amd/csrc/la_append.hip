// Device-side latent-cache append with query RoPE (la_append_kv).
//
// Replaces LatentKVCache::append_host (paths relative to the reference repo,
// src/mla_config.cuh:57-72), which copies one host row into the cache with two
// host-to-device copies and a stream synchronize per token and keeps the
// length on the host. Here one launch (two for prompts) appends tokens_per_seq
// rows to every sequence of a batch, the lengths live in device memory, and nothing waits on
// the host, so a decode step (append -> absorb -> attend -> project) is one
// stream-ordered sequence of kernels.
//
// Rows are stored as the reference's cache holds them: [c_t | k_rope] with
// k_rope not rotated (the attention rotates keys by position,
// src/fused_mla.cu:34-54). The reference never rotates the query; this kernel
// rotates q_rope for the query's own position with the same rotate-half
// pairing (i, i + dR/2) and the same tables (src/fused_mla.cu:43-51), so
// callers no longer pre-rotate it.
#include "la_internal.hpp"

#include <algorithm>

namespace la {
namespace {

constexpr int kAppendThreads = 1024;
constexpr int kFillThreads = 256;

__device__ inline void store_any(void* base, int dtype, int64_t i, float v) {
  if (dtype == LA_DTYPE_BF16) reinterpret_cast<__hip_bfloat16*>(base)[i] = __float2bfloat16(v);
  else if (dtype == LA_DTYPE_F16) reinterpret_cast<__half*>(base)[i] = __float2half(v);
  else if (dtype == LA_DTYPE_FP8_E4M3) reinterpret_cast<uint8_t*>(base)[i] = f32_to_fp8(v);
  else reinterpret_cast<float*>(base)[i] = v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// Eight consecutive elements as f32, and back; i is a multiple of 8 and the
// base is aligned for the vector (append_vec).
__device__ inline void load8(const void* base, int dtype, int64_t i, float (&v)[8]) {
  if (dtype == LA_DTYPE_F32) {
    const f32x4* q = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + i);
    const f32x4 a = q[0], b = q[1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else if (dtype == LA_DTYPE_FP8_E4M3) {
    const u32x2 q = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint8_t*>(base) + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = fp8_to_f32((q[e >> 2] >> (8 * (e & 3))) & 0xFF);
  } else {
    const u16x8 q = *reinterpret_cast<const u16x8*>(reinterpret_cast<const uint16_t*>(base) + i);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = dtype == LA_DTYPE_BF16 ? __bfloat162float(__builtin_bit_cast(__hip_bfloat16, (uint16_t)q[e]))
                                    : __half2float(__builtin_bit_cast(__half, (uint16_t)q[e]));
  }
}
__device__ inline void store8(void* base, int dtype, int64_t i, const float (&v)[8]) {
  if (dtype == LA_DTYPE_F32) {
    f32x4* q = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(base) + i);
    q[0] = f32x4{v[0], v[1], v[2], v[3]};
    q[1] = f32x4{v[4], v[5], v[6], v[7]};
  } else if (dtype == LA_DTYPE_FP8_E4M3) {
    u32x2 q = {0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e >> 2] |= (uint32_t)f32_to_fp8(v[e]) << (8 * (e & 3));
    *reinterpret_cast<u32x2*>(reinterpret_cast<uint8_t*>(base) + i) = q;
  } else {
    u16x8 q;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      q[e] = dtype == LA_DTYPE_BF16 ? __builtin_bit_cast(uint16_t, __float2bfloat16(v[e]))
                                    : __builtin_bit_cast(uint16_t, __float2half(v[e]));
    *reinterpret_cast<u16x8*>(reinterpret_cast<uint16_t*>(base) + i) = q;
  }
}

// Length of sequence s and the row of its first new token (-1: no room; a
// paged cache is a virtual region of blocks_per_seq blocks, mapped per row).
__device__ inline int64_t append_row0(const AppendProblem& p, int s, int* len) {
  const int64_t start = p.block_table ? 0 : p.offsets ? (int64_t)p.offsets[s] : (int64_t)s * p.capacity;
  const int64_t end = p.block_table ? (int64_t)p.blocks_per_seq * p.block_size
                      : p.offsets   ? (int64_t)p.offsets[s + 1]
                                    : start + p.capacity;
  *len = p.lens[s];
  const bool ok = start >= 0 && start <= end && (p.block_table || end <= p.total_rows) && *len >= 0 &&
                  (int64_t)*len + p.tokens <= end - start;
  return ok ? start + *len : -1;
}

// Threads t0, t0 + step, ... of sequence s: its new rows, and its query pairs.
// Index arithmetic is 32-bit unsigned (the entry point keeps the per-sequence
// counts below 2^31, a step is at most 2^20).
// kVec: eight elements of a row per thread (append_vec), else one. The
// rotation takes four consecutive pairs per thread with 16-B loads when dR/2
// is a multiple of 4 (every query row and table row is then 16-B aligned; the
// entry point checks the base pointers), one pair otherwise.
template <bool kVec>
__device__ inline void append_part(const AppendProblem& p, int s, int64_t row0, int len, uint32_t t0, uint32_t step) {
  constexpr int kE = kVec ? 8 : 1;
  const int row = p.dc + p.dR;
  const uint32_t per = row / kE;
  const uint32_t n = p.tokens * per;
  const int64_t tok0 = (int64_t)s * p.tokens;
  for (uint32_t i = t0; i < n; i += step) {
    const int t = i / per;
    const int c = kE * (i - t * per);
    int64_t dst = row0 + t;
    if (p.block_table) {  // position len + t of sequence s in the pool (block id clamped into it)
      const int64_t pos = (int64_t)len + t;
      int64_t b = p.block_table[(int64_t)s * p.blocks_per_seq + pos / p.block_size];
      b = b < 0 ? 0 : (b >= p.pool_blocks ? p.pool_blocks - 1 : b);
      dst = b * p.block_size + pos % p.block_size;
    }
    const void* const src = c < p.dc ? p.c_t : p.k_rope;
    const int64_t at = c < p.dc ? (tok0 + t) * p.dc + c : (tok0 + t) * p.dR + (c - p.dc);
    if constexpr (kVec) {
      float v[8];
      load8(src, p.src_dtype, at, v);
      store8(p.kv, p.kv_dtype, dst * row + c, v);
    } else {
      store_any(p.kv, p.kv_dtype, dst * row + c, load_any(src, p.src_dtype, at));
    }
  }

  if (!p.q_rope) return;
  // query j of this sequence is the token at position len + tokens - qps + j
  const int half = p.dR >> 1;
  float* const qs = p.q_rope + (int64_t)s * p.qps * p.nh * p.dR;
  const int pos_base = len + p.tokens - p.qps;
  if ((half & 3) == 0) {
    const uint32_t quads = half >> 2;
    const uint32_t nq = p.qps * p.nh * quads;
    for (uint32_t i = t0; i < nq; i += step) {
      const int qr = i / quads;  // j * nh + h
      const int e = 4 * (i - qr * quads);
      int64_t pos = pos_base + qr / p.nh;
      if (p.rope_rows > 0 && pos >= p.rope_rows) pos = p.rope_rows - 1;
      f32x4* q0 = reinterpret_cast<f32x4*>(qs + (int64_t)qr * p.dR + e);
      f32x4* q1 = reinterpret_cast<f32x4*>(qs + (int64_t)qr * p.dR + e + half);
      const f32x4 x = *q0, y = *q1;
      const f32x4 cs = *reinterpret_cast<const f32x4*>(p.rope_cos + pos * half + e);
      const f32x4 sn = *reinterpret_cast<const f32x4*>(p.rope_sin + pos * half + e);
      *q0 = x * cs - y * sn;
      *q1 = x * sn + y * cs;
    }
  } else {
    const uint32_t nq = (uint32_t)(p.qps * p.nh) * half;
    for (uint32_t i = t0; i < nq; i += step) {
      const int qr = i / (uint32_t)half;
      const int e = i - qr * half;
      int64_t pos = pos_base + qr / p.nh;
      if (p.rope_rows > 0 && pos >= p.rope_rows) pos = p.rope_rows - 1;
      float* q = qs + (int64_t)qr * p.dR;
      const float x = q[e], y = q[e + half];
      const float cs = p.rope_cos[pos * half + e], sn = p.rope_sin[pos * half + e];
      q[e] = x * cs - y * sn;
      q[e + half] = x * sn + y * cs;
    }
  }
}

// One workgroup per sequence: every thread reads the sequence's length, copies
// (and converts) its share of the new rows and rotates its share of the query
// pairs; after a barrier (all reads of the old length done) thread 0 stores
// the new length. A sequence without room is left untouched and raises
// *status. With up to 1024 elements and groups of 4 query pairs (a decode step
// at 128 heads) every thread has one of each, so a sequence costs one memory
// round trip for its loads and one for its stores.
template <bool kVec>
__global__ __launch_bounds__(kAppendThreads) void append_kernel(AppendProblem p) {
  const int s = blockIdx.x;
  int len;
  const int64_t row0 = append_row0(p, s, &len);
  if (row0 < 0) {
    if (threadIdx.x == 0 && p.status) *p.status = 1;
    return;
  }
  append_part<kVec>(p, s, row0, len, threadIdx.x, kAppendThreads);
  __syncthreads();
  if (threadIdx.x == 0) p.lens[s] = len + p.tokens;
}

// Prompts: blocks_per workgroups per sequence, which leave the lengths to a
// second launch (append_lens_kernel), since each of them reads the old one.
// Memory-bound: 8 x 1021 bf16 rows (18.8 MB read and written) in 7.3 us,
// against 306 with one workgroup per sequence and 2-B accesses.
template <bool kVec>
__global__ __launch_bounds__(kFillThreads) void append_rows_kernel(AppendProblem p, int blocks_per) {
  const int s = blockIdx.x / blocks_per;
  const int b = blockIdx.x - s * blocks_per;
  int len;
  const int64_t row0 = append_row0(p, s, &len);
  if (row0 < 0) return;
  append_part<kVec>(p, s, row0, len, b * kFillThreads + threadIdx.x, blocks_per * kFillThreads);
}
__global__ __launch_bounds__(kFillThreads) void append_lens_kernel(AppendProblem p) {
  const int s = blockIdx.x * kFillThreads + threadIdx.x;
  if (s >= p.num_seqs) return;
  int len;
  if (append_row0(p, s, &len) >= 0) p.lens[s] = len + p.tokens;
  else if (p.status) *p.status = 1;
}

// Eight elements per thread: whole groups in both parts of a row, and every
// base aligned for their loads and stores.
bool append_vec(const AppendProblem& p) {
  const auto aligned = [](const void* q, int dtype) {
    return (reinterpret_cast<uintptr_t>(q) & (dtype == LA_DTYPE_FP8_E4M3 ? 7 : 15)) == 0;
  };
  return p.dc % 8 == 0 && p.dR % 8 == 0 && aligned(p.kv, p.kv_dtype) && aligned(p.c_t, p.src_dtype) &&
         aligned(p.k_rope, p.src_dtype);
}

}  // namespace

hipError_t launch_append(const AppendProblem& p, hipStream_t stream) {
  if (p.num_seqs == 0) return hipSuccess;
  // One element per thread while that is one round (a decode step's token), or,
  // into an FP8 cache, one and a half: the software conversions of eight in one
  // thread are a longer chain (64 sequences, FP8 from fp32 with a fill launch, one
  // against eight elements per thread: 2 tokens of 576 4.70 / 5.04 us, 3 tokens
  // 5.05 / 5.06, 4 tokens with rotated queries 6.40 / 5.98, 5 tokens 5.85 / 5.25;
  // bf16 2 tokens 4.83 / 4.42).
  const int64_t elems = (int64_t)p.tokens * (p.dc + p.dR);
  const bool vec = 2 * elems > (p.kv_dtype == LA_DTYPE_FP8_E4M3 ? 3 : 2) * kAppendThreads && append_vec(p);
  const int half = p.dR / 2;
  const int64_t rows_n = elems / (vec ? 8 : 1);
  const int64_t quer_n = p.q_rope ? (int64_t)p.qps * p.nh * (half % 4 == 0 ? half / 4 : half) : 0;
  const int64_t n = std::max(rows_n, quer_n);
  // One workgroup per sequence up to four rounds of it (56 new rows of 576
  // elements): a second launch costs what about two rounds do.
  if (n <= 4 * kAppendThreads) {
    auto k = vec ? append_kernel<true> : append_kernel<false>;
    hipLaunchKernelGGL(k, dim3((unsigned)p.num_seqs), dim3(kAppendThreads), 0, stream, p);
    return hipGetLastError();
  }
  // enough workgroups for one round, up to 16 per CU of a 256-CU device in all
  const int64_t want = (n + kFillThreads - 1) / kFillThreads;
  const int64_t most = std::max<int64_t>(4096 / p.num_seqs, 1);
  const int per = (int)std::min(want, most);
  auto k = vec ? append_rows_kernel<true> : append_rows_kernel<false>;
  hipLaunchKernelGGL(k, dim3((unsigned)((int64_t)p.num_seqs * per)), dim3(kFillThreads), 0, stream, p, per);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(append_lens_kernel, dim3((unsigned)((p.num_seqs + kFillThreads - 1) / kFillThreads)),
                     dim3(kFillThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace la
