// Decompress-then-attend MLA on the GPU (la_naive_mla): the reference's naive
// path (paths relative to the reference repo: src/naive_mla.cu:91-245 and the
// PyTorch restatement tests/test_python.py:26-63) computed the way its math
// reads, independently of the absorbed kernels:
//   K_nope = c_t . W_UK^T   (S, nh*dn)      V = c_t . W_UV^T   (S, nh*dv)
//   s[h,pos] = scale*(q_nope[h] . K_nope[pos,h] + q_rope[h] . RoPE(k_rope[pos], pos))
//   out[h]   = softmax_pos(s[h]) . V[:,h]
// in fp32 from the 16-bit (or fp32) cache and weights. The reference's cuBLAS
// call reads K/V transposed; this path does not reproduce that.
//
// 16-bit caches with weights of the same type and 128-dim heads decompress on
// the matrix cores (products of 16-bit values are exact in fp32, sums are
// fp32) and K_nope and V are used where they are made, never stored: a
// workgroup decompresses 256 positions of one head and either dots them with
// the head's query (naive_k_kernel) or weights and sums them
// (naive_v_kernel). At S = 8192 and 128 heads the two products are 275 GFLOP:
// 157 to 172 us each (0.8 to 0.87 PFLOP/s; matrix cores busy half of it), 329 us
// a call with the rest.
// Other types and shapes take the plain kernels: a 64x64-tiled VALU GEMM into
// fp32 K_nope and V, one thread per (head, position) for the scores, one
// workgroup per head for the softmax and the weighted sum (10.2 ms there).
#include "la_internal.hpp"

namespace la {
namespace {

constexpr int kTile = 64;  // output tile of the decompression GEMM
constexpr int kKStep = 16;

// Y[r][n] = sum_c X[r][c] * W[n][c] for r < rows, n < N, c < K. X rows have
// stride ldx elements (the cache row), W rows stride K. 256 threads, each
// 4 x 4 outputs; X and W tiles staged through LDS transposed ([c][r]).
template <typename XT, typename WT>
__global__ __launch_bounds__(256) void decompress_kernel(const XT* __restrict__ X, int ldx, const WT* __restrict__ W,
                                                         float* __restrict__ Y, int rows, int N, int K) {
  __shared__ float xs[kKStep][kTile + 4];
  __shared__ float ws[kKStep][kTile + 4];
  const int r0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  float acc[4][4] = {};
  for (int c0 = 0; c0 < K; c0 += kKStep) {
    for (int i = threadIdx.x; i < kTile * kKStep; i += 256) {
      const int rr = i / kKStep, cc = i % kKStep;
      const int r = r0 + rr, n = n0 + rr, c = c0 + cc;
      xs[cc][rr] = (r < rows && c < K) ? to_f32(X[(int64_t)r * ldx + c]) : 0.f;
      ws[cc][rr] = (n < N && c < K) ? to_f32(W[(int64_t)n * K + c]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int cc = 0; cc < kKStep; ++cc) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = xs[cc][ty + 16 * i];
        b[i] = ws[cc][tx + 16 * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + ty + 16 * i;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n < N) Y[(int64_t)r * N + n] = acc[i][j];
    }
  }
}

// s[h][pos] for one query: thread per (pos, head), RoPE of the key by its
// position (rotate-half, src/fused_mla.cu:43-51; positions past the table use
// its last row).
template <typename KT>
__global__ __launch_bounds__(256) void naive_scores_kernel(const KT* __restrict__ kv, int S, int dc, int dR,
                                                           const float* __restrict__ Kn, int nh, int dn,
                                                           const float* __restrict__ q_nope,
                                                           const float* __restrict__ q_rope,
                                                           const float* __restrict__ cos_t,
                                                           const float* __restrict__ sin_t, int64_t rope_rows,
                                                           float scale, float* __restrict__ scores) {
  const int pos = blockIdx.x * 256 + threadIdx.x;
  const int h = blockIdx.y;
  if (pos >= S) return;
  const float* k = Kn + ((int64_t)pos * nh + h) * dn;
  const float* q = q_nope + (int64_t)h * dn;
  float a = 0.f;
  for (int i = 0; i < dn; ++i) a += q[i] * k[i];
  const int half = dR >> 1;
  const int64_t r = (rope_rows > 0 && pos >= rope_rows) ? rope_rows - 1 : pos;
  const KT* kr = kv + (int64_t)pos * (dc + dR) + dc;
  const float* qr = q_rope + (int64_t)h * dR;
  float b = 0.f;
  for (int i = 0; i < half; ++i) {
    const float k0 = to_f32(kr[i]), k1 = to_f32(kr[i + half]);
    const float c = cos_t[r * half + i], s = sin_t[r * half + i];
    b += qr[i] * (k0 * c - k1 * s) + qr[i + half] * (k0 * s + k1 * c);
  }
  scores[(int64_t)h * S + pos] = scale * a + scale * b;
}

// out[h][j] = sum_pos softmax(s[h])[pos] * V[pos][h*dv + j]: one workgroup per
// head; max and sum reduced over the workgroup, then thread j < dv sums over
// positions.
__global__ __launch_bounds__(256) void naive_softmax_pv_kernel(const float* __restrict__ scores, int S,
                                                               const float* __restrict__ V, int nh, int dv,
                                                               float* __restrict__ out) {
  const int h = blockIdx.x;
  const float* s = scores + (int64_t)h * S;
  __shared__ float red[8];
  __shared__ float stat[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (S == 0) {  // empty cache: zero output (as the absorbed path gives)
    for (int j = tid; j < dv; j += 256) out[(int64_t)h * dv + j] = 0.f;
    return;
  }
  float m = -INFINITY;
  for (int p = tid; p < S; p += 256) m = fmaxf(m, s[p]);
  m = wave_max(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  if (tid == 0) stat[0] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  m = stat[0];
  float l = 0.f;
  for (int p = tid; p < S; p += 256) l += expf(s[p] - m);
  l = wave_sum(l);
  if (lane == 0) red[4 + wave] = l;
  __syncthreads();
  if (tid == 0) stat[1] = (red[4] + red[5]) + (red[6] + red[7]);
  __syncthreads();
  const float inv_l = 1.f / stat[1];
  for (int j = tid; j < dv; j += 256) {
    float acc = 0.f;
    for (int p = 0; p < S; ++p) acc += expf(s[p] - m) * V[((int64_t)p * nh + h) * dv + j];
    out[(int64_t)h * dv + j] = acc * inv_l;
  }
}

template <typename XT, typename WT>
hipError_t decompress(const NaiveProblem& p, const void* W, float* Y, int N, hipStream_t stream) {
  const dim3 grid((unsigned)((N + kTile - 1) / kTile), (unsigned)((p.S + kTile - 1) / kTile));
  hipLaunchKernelGGL((decompress_kernel<XT, WT>), grid, dim3(256), 0, stream, reinterpret_cast<const XT*>(p.kv),
                     p.dc + p.dR, reinterpret_cast<const WT*>(W), Y, p.S, N, p.dc);
  return hipGetLastError();
}

template <typename XT>
hipError_t decompress_w(const NaiveProblem& p, const void* W, int wdt, float* Y, int N, hipStream_t stream) {
  if (wdt == LA_DTYPE_BF16) return decompress<XT, __hip_bfloat16>(p, W, Y, N, stream);
  if (wdt == LA_DTYPE_F16) return decompress<XT, __half>(p, W, Y, N, stream);
  return decompress<XT, float>(p, W, Y, N, stream);
}

template <typename KT>
hipError_t run_naive_t(const NaiveProblem& p, hipStream_t stream) {
  if (p.S == 0) {
    hipLaunchKernelGGL(naive_softmax_pv_kernel, dim3((unsigned)p.nh), dim3(256), 0, stream, p.scores, 0, p.V, p.nh,
                       p.dv, p.out);
    return hipGetLastError();
  }
  hipError_t e = decompress_w<KT>(p, p.W_UK, p.wuk_dtype, p.Kn, p.nh * p.dn, stream);
  if (e == hipSuccess) e = decompress_w<KT>(p, p.W_UV, p.wuv_dtype, p.V, p.nh * p.dv, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(naive_scores_kernel<KT>, dim3((unsigned)((p.S + 255) / 256), (unsigned)p.nh), dim3(256), 0,
                     stream, reinterpret_cast<const KT*>(p.kv), p.S, p.dc, p.dR, p.Kn, p.nh, p.dn, p.q_nope,
                     p.q_rope, p.rope_cos, p.rope_sin, p.rope_rows, p.scale, p.scores);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(naive_softmax_pv_kernel, dim3((unsigned)p.nh), dim3(256), 0, stream, p.scores, p.S, p.V, p.nh,
                     p.dv, p.out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Matrix-core path
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) char lchar;

template <typename T>
struct Mm;
template <>
struct Mm<__hip_bfloat16> {
  typedef bf16x8 vec;
  static __device__ inline f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mm<__half> {
  typedef f16x8 vec;
  static __device__ inline f32x16 mma(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

constexpr int kHd = 128;      // head dim (nope or value): one workgroup's weight rows
constexpr int kPos = 256;     // positions per workgroup
constexpr int kBk = 32;       // latent columns per stage
constexpr int kStages = 3;    // one computed, two in flight
constexpr int kMmThreads = 512;
// a stage: position rows, then weight rows, 64 B each; chunk j of row r at j ^ sw(r)
constexpr int kStageBytes = (kPos + kHd) * kBk * 2;
__device__ inline int sw(int r) { return (r >> 2) & 3; }
// acc[i][j] of wave (wa, wb) = rows 64 wa + 32 i of the M operand times rows
// 64 wb + 32 j of the N operand, over K columns; the M operand is the weights
// (kWeightsM) or the positions. Every stage is three 1-KB HBM->LDS copies per
// wave (16 rows of 64 B each, the chunk permutation applied to the addresses
// read); two stages stay in flight behind the one computed, one barrier each.
// 72 KB of LDS and under 128 VGPRs: two workgroups per CU, so one's fill and
// epilogue run under the other's products.
template <typename T, bool kWeightsM>
__device__ inline void tile_product(const char* X, int64_t ldx, int rows, const char* W, int K, lchar* L, int wave,
                                    int lane, f32x16 (&acc)[2][2]) {
  typedef typename Mm<T>::vec vec;
  const int rr = lane >> 2, ch = lane & 3;
  // copies c = 3 wave + i: 16 position rows (c < 16) or weight rows
  const char* src[3];
  int dst[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int c = 3 * wave + i;
    const int r = 16 * c + rr;
    src[i] = (c < 16 ? X + (int64_t)min(r, rows - 1) * ldx : W + (int64_t)(r - kPos) * K * 2) + 16 * (ch ^ sw(r));
    dst[i] = 1024 * c;
  }
  const int stages = K / kBk;
  auto issue = [&](int k) {
    const int buf = (k % kStages) * kStageBytes;
    const int kk = min(k, stages - 1);  // past the end: the last stage again, never read
#pragma unroll
    for (int i = 0; i < 3; ++i)
      __builtin_amdgcn_global_load_lds(src[i] + (int64_t)kk * kBk * 2, (lds_void*)(L + buf + dst[i]), 16, 0, 0);
  };
  const int wm = wave & 1, wn = wave >> 1;  // weight half, position quarter
  const int r32 = lane & 31, hi = lane >> 5;
  issue(0);
  issue(1);
  for (int k = 0; k < stages; ++k) {
    __builtin_amdgcn_s_waitcnt(0x0F73);  // vmcnt(3): this wave's copies of stage k have landed
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // everyone's; stage k - 1 is read
    issue(k + 2);
    const lchar* S = L + (k % kStages) * kStageBytes;
#pragma unroll
    for (int ks = 0; ks < kBk / 16; ++ks) {
      vec w[2], x[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rw = kPos + 64 * wm + 32 * i + r32, rx = 64 * wn + 32 * i + r32;
        w[i] = *reinterpret_cast<const __attribute__((address_space(3))) vec*>(S + rw * 64 + 16 * ((2 * ks + hi) ^ sw(rw)));
        x[i] = *reinterpret_cast<const __attribute__((address_space(3))) vec*>(S + rx * 64 + 16 * ((2 * ks + hi) ^ sw(rx)));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = kWeightsM ? Mm<T>::mma(w[i], x[j], acc[i][j]) : Mm<T>::mma(x[i], w[j], acc[i][j]);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the copies past the end have landed
  // 16 wait states (and more instructions) before the accumulators' first VALU reader
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) asm volatile("s_nop 15" : "+v"(acc[i][j]));
  asm volatile("s_barrier" ::: "memory");  // the stages are reused by the epilogue
}

// Workgroup id -> (head, position block): an XCD (id % 8) takes every eighth
// head and goes through them per position block, so its weights (16 heads: 2
// MB) stay in its L2 and each block's cache rows are fetched once.
__device__ inline bool mm_coords(int nh, int* h, int* pb) {
  const int nh8 = (nh + 7) / 8, x = blockIdx.x & 7, k = blockIdx.x >> 3;
  *h = x + 8 * (k % nh8);
  *pb = k / nh8;
  return *h < nh;
}

// scores[h][pos] += scale * (q_nope[h] . K_nope[pos,h]) (the rope part is there already)
template <typename T>
__global__ __launch_bounds__(kMmThreads, 4) void naive_k_kernel(const T* __restrict__ kv, int S, int dc, int dR,
                                                                const T* __restrict__ W, int nh,
                                                                const float* __restrict__ q_nope, float scale,
                                                                float* __restrict__ scores) {
  extern __shared__ __attribute__((aligned(1024))) char mm_lds[];
  lchar* const L = (lchar*)mm_lds;
  int h, pb;
  if (!mm_coords(nh, &h, &pb)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ldx = (dc + dR) * 2;
  f32x16 acc[2][2] = {};
  tile_product<T, true>(reinterpret_cast<const char*>(kv) + (int64_t)pb * kPos * ldx, ldx, S - pb * kPos,
                        reinterpret_cast<const char*>(W) + (int64_t)h * kHd * dc * 2, dc, L, wave, lane, acc);
  // lane: position 64 wn + 32 j + lane%32; register e of block i: K column 64 wm + 32 i + 8 (e/4) + 4 (lane/32) + e%4
  const int wm = wave & 1, wn = wave >> 1;
  float a[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(q_nope + h * kHd + 64 * wm + 32 * i + 8 * e4 + 4 * (lane >> 5));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 2; ++j) a[j] += acc[i][j][4 * e4 + e] * q[e];
    }
  __attribute__((address_space(3))) float* part = reinterpret_cast<__attribute__((address_space(3))) float*>(L);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float v = sum_halves(a[j]);
    if (lane < 32) part[kPos * wm + 64 * wn + 32 * j + lane] = v;
  }
  __syncthreads();
  const int pos = pb * kPos + threadIdx.x;
  if (threadIdx.x < kPos && pos < S) {
    float* const d = scores + (int64_t)h * S + pos;
    *d = scale * (part[threadIdx.x] + part[kPos + threadIdx.x]) + *d;
  }
}

// part[pb][h][j] = sum over the block's positions of e[h][pos] V[pos,h,j]
template <typename T>
__global__ __launch_bounds__(kMmThreads, 4) void naive_v_kernel(const T* __restrict__ kv, int S, int dc, int dR,
                                                                const T* __restrict__ W, int nh,
                                                                const float* __restrict__ e_in,
                                                                float* __restrict__ part_out) {
  extern __shared__ __attribute__((aligned(1024))) char mm_lds[];
  lchar* const L = (lchar*)mm_lds;
  int h, pb;
  if (!mm_coords(nh, &h, &pb)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ldx = (dc + dR) * 2;
  const int pos = pb * kPos + threadIdx.x;
  const float ev = threadIdx.x < kPos && pos < S ? e_in[(int64_t)h * S + pos] : 0.f;
  f32x16 acc[2][2] = {};
  tile_product<T, false>(reinterpret_cast<const char*>(kv) + (int64_t)pb * kPos * ldx, ldx, S - pb * kPos,
                         reinterpret_cast<const char*>(W) + (int64_t)h * kHd * dc * 2, dc, L, wave, lane, acc);
  typedef __attribute__((address_space(3))) float lfloat;
  lfloat* es = reinterpret_cast<lfloat*>(L);
  lfloat* red = es + kPos;  // [position quarter][V column]
  if (threadIdx.x < kPos) es[threadIdx.x] = ev;
  __syncthreads();
  // lane: V column 64 wm + 32 j + lane%32; register e of block i: position 64 wn + 32 i + 8 (e/4) + 4 (lane/32) + e%4
  const int wm = wave & 1, wn = wave >> 1;
  float a[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const f32x4 w = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(
          es + 64 * wn + 32 * i + 8 * e4 + 4 * (lane >> 5));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 2; ++j) a[j] += acc[i][j][4 * e4 + e] * w[e];
    }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float v = sum_halves(a[j]);
    if (lane < 32) red[kHd * wn + 64 * wm + 32 * j + lane] = v;
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < kHd)
    part_out[((int64_t)pb * nh + h) * kHd + t] = (red[t] + red[kHd + t]) + (red[2 * kHd + t] + red[3 * kHd + t]);
}

// scores[h][pos] = scale * (q_rope[h] . RoPE(k_rope[pos], pos)): lane = position,
// its rotated key in registers, the query through scalar loads; a wave takes
// every fourth head of its share (heads blockIdx.y * kRopeHeads ..).
constexpr int kRopeHeads = 32;
template <typename KT>
__global__ __launch_bounds__(256) void naive_rope_kernel(const KT* __restrict__ kv, int S, int dc, int nh,
                                                         const float* __restrict__ q_rope,
                                                         const float* __restrict__ cos_t,
                                                         const float* __restrict__ sin_t, int64_t rope_rows, float scale,
                                                         float* __restrict__ scores) {
  constexpr int dR = 64;
  const int pos = blockIdx.x * 64 + (threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int pc = min(pos, S - 1);
  const int64_t r = (rope_rows > 0 && pc >= rope_rows) ? rope_rows - 1 : pc;
  const KT* kr = kv + (int64_t)pc * (dc + dR) + dc;
  float k[dR];
#pragma unroll
  for (int i = 0; i < dR / 2; ++i) {
    const float k0 = to_f32(kr[i]), k1 = to_f32(kr[i + dR / 2]);
    const float c = cos_t[r * (dR / 2) + i], s = sin_t[r * (dR / 2) + i];
    k[i] = k0 * c - k1 * s;
    k[i + dR / 2] = k0 * s + k1 * c;
  }
  const int h_end = min(nh, ((int)blockIdx.y + 1) * kRopeHeads);
  for (int h = blockIdx.y * kRopeHeads + wave; h < h_end; h += 4) {
    const float* q = q_rope + (int64_t)h * dR;
    float b0 = 0.f, b1 = 0.f;
#pragma unroll
    for (int i = 0; i < dR; i += 2) {
      b0 += q[i] * k[i];
      b1 += q[i + 1] * k[i + 1];
    }
    if (pos < S) scores[(int64_t)h * S + pos] = scale * (b0 + b1);
  }
}

// scores[h] -> e = exp(s - max), in place, and inv_l[h] = 1 / sum e. One workgroup per head.
__global__ __launch_bounds__(1024) void naive_softmax_kernel(float* __restrict__ scores, int S, float* __restrict__ inv_l) {
  float* s = scores + (int64_t)blockIdx.x * S;
  __shared__ float red[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float m = -INFINITY;
  for (int p = tid; p < S; p += 1024) m = fmaxf(m, s[p]);
  m = wave_max(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int w = 1; w < 16; ++w) m = fmaxf(m, red[w]);
  __syncthreads();
  float l = 0.f;
  for (int p = tid; p < S; p += 1024) {
    const float e = expf(s[p] - m);
    s[p] = e;
    l += e;
  }
  l = wave_sum(l);
  if (lane == 0) red[wave] = l;
  __syncthreads();
  if (tid == 0) {
    float t = 0.f;
    for (int w = 0; w < 16; ++w) t += red[w];
    inv_l[blockIdx.x] = 1.f / t;
  }
}

// out[h][j] = inv_l[h] * sum of the position blocks' parts; 4 threads per column
__global__ __launch_bounds__(4 * kHd) void naive_sum_kernel(const float* __restrict__ part, int blocks, int nh,
                                                            const float* __restrict__ inv_l, float* __restrict__ out) {
  const int h = blockIdx.x, j = threadIdx.x & (kHd - 1), q = threadIdx.x / kHd;
  __shared__ float red[4][kHd];
  float a = 0.f;
  for (int b = q; b < blocks; b += 4) a += part[((int64_t)b * nh + h) * kHd + j];
  red[q][j] = a;
  __syncthreads();
  if (q == 0) out[(int64_t)h * kHd + j] = ((red[0][j] + red[1][j]) + (red[2][j] + red[3][j])) * inv_l[h];
}

bool naive_mm_supported(const NaiveProblem& p) {
  const auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return p.S > 0 && (p.kv_dtype == LA_DTYPE_BF16 || p.kv_dtype == LA_DTYPE_F16) && p.wuk_dtype == p.kv_dtype &&
         p.wuv_dtype == p.kv_dtype && p.dn == kHd && p.dv == kHd && p.dR == 64 && p.dc % (2 * kBk) == 0 &&
         aligned(p.kv) && aligned(p.W_UK) && aligned(p.W_UV) && aligned(p.q_nope) && device_is_gfx950();
}

// Workspace: inv_l in the place of K_nope, the position blocks' parts in V's.
template <typename T>
hipError_t run_naive_mm(const NaiveProblem& p, hipStream_t stream) {
  constexpr int lds = kStages * kStageBytes;
  static OncePerDevice once_k, once_v;
  hipError_t e = allow_lds(once_k, reinterpret_cast<const void*>(&naive_k_kernel<T>), lds);
  if (e == hipSuccess) e = allow_lds(once_v, reinterpret_cast<const void*>(&naive_v_kernel<T>), lds);
  if (e != hipSuccess) return e;
  const int blocks = (p.S + kPos - 1) / kPos;
  const T* kv = reinterpret_cast<const T*>(p.kv);
  const dim3 rgrid((unsigned)((p.S + 63) / 64), (unsigned)((p.nh + kRopeHeads - 1) / kRopeHeads));
  const dim3 grid((unsigned)(8 * ((p.nh + 7) / 8) * blocks));
  hipLaunchKernelGGL(naive_rope_kernel<T>, rgrid, dim3(256), 0, stream, kv, p.S, p.dc, p.nh, p.q_rope, p.rope_cos,
                     p.rope_sin, p.rope_rows, p.scale, p.scores);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(naive_k_kernel<T>, grid, dim3(kMmThreads), lds, stream, kv, p.S, p.dc, p.dR,
                     reinterpret_cast<const T*>(p.W_UK), p.nh, p.q_nope, p.scale, p.scores);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(naive_softmax_kernel, dim3((unsigned)p.nh), dim3(1024), 0, stream, p.scores, p.S, p.Kn);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(naive_v_kernel<T>, grid, dim3(kMmThreads), lds, stream, kv, p.S, p.dc, p.dR,
                     reinterpret_cast<const T*>(p.W_UV), p.nh, p.scores, p.V);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(naive_sum_kernel, dim3((unsigned)p.nh), dim3(4 * kHd), 0, stream, p.V, blocks, p.nh, p.Kn, p.out);
  return hipGetLastError();
}

}  // namespace

size_t naive_workspace_bytes(int64_t S, int nh, int dn, int dv) {
  const auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  return up((size_t)S * nh * dn * 4) + up((size_t)S * nh * dv * 4) + up((size_t)S * nh * 4);
}

hipError_t launch_naive(NaiveProblem p, void* workspace, hipStream_t stream) {
  const auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  char* w = static_cast<char*>(workspace);
  p.Kn = reinterpret_cast<float*>(w);
  p.V = reinterpret_cast<float*>(w + up((size_t)p.S * p.nh * p.dn * 4));
  p.scores = reinterpret_cast<float*>(w + up((size_t)p.S * p.nh * p.dn * 4) + up((size_t)p.S * p.nh * p.dv * 4));
  if (naive_mm_supported(p))
    return p.kv_dtype == LA_DTYPE_BF16 ? run_naive_mm<__hip_bfloat16>(p, stream) : run_naive_mm<__half>(p, stream);
  if (p.kv_dtype == LA_DTYPE_BF16) return run_naive_t<__hip_bfloat16>(p, stream);
  if (p.kv_dtype == LA_DTYPE_F16) return run_naive_t<__half>(p, stream);
  if (p.kv_dtype == LA_DTYPE_FP8_E4M3) return run_naive_t<fp8e4m3>(p, stream);
  return run_naive_t<float>(p, stream);
}

}  // namespace la
