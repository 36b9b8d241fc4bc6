// MFMA split-KV MLA decode kernel with 16 query heads per workgroup, for few
// heads or little work per compute unit. Same operation, cache types, split
// plan and partial slots as decode_mfma_kernel (la_mfma.hip), which keeps 128
// heads and one wave per SIMD: the best rate once its workgroups stream many
// tiles, but with 16 heads it still runs the matrix work of 128, and its
// prologue and epilogue (25K cycles) are most of its time on a few tiles.
//
// A workgroup of kW waves walks tiles of 16 kW positions on
// v_mfma_f32_16x16x32. Per tile:
//   * Staging: wave w copies rows 16w .. 16w+15. 16-bit c_t rows go HBM->LDS
//     directly (one 1-KB copy a row); FP8 rows come through registers and are
//     expanded to bf16. The k_rope part is loaded into registers with its cos
//     and sin rows, rotated there and written to LDS.
//   * Scores: S^T[16 positions x 16 heads] per wave, A = the wave's own rows
//     (so no barrier yet), B = Q (18 k-steps, in registers for the segment).
//   * Softmax: the waves' maxima meet in LDS, every wave then knows the tile's
//     running maximum m per head; P = 2^(s - m) goes to LDS as the 16-bit B
//     operand, O and the running sum are rescaled where m moved.
//   * PV: wave w holds O^T for 512 / kW latent columns (lane = head): A =
//     value rows transposed by ds_read_b64_tr_b16, B = P.
// There is one tile buffer and no pipeline across tiles: with kW = 4 two
// workgroups share a CU (165 VGPRs, 76 KB of LDS) and one's loads run under
// the other's compute; kW = 8 takes twice the positions per memory round trip
// for launches of at most one workgroup per CU, where latency is all there is
// (128-row chunks are one tile).
//
// LDS rows are unpadded (two workgroups per CU leave no room for padding):
// the 16-B chunk j of c_t row r sits at j ^ cf(r), which spreads both the
// score reads (16 rows at one chunk) and the transposed value reads (8 rows x
// 32 B per half wave) over all banks. The copies write LDS linearly, so the
// permutation is applied to the global address each lane reads.
//
// What bounds it: memory latency on short chunks; at 16 heads and long chunks
// its stream (151 MB in 33 us with a fixed part of about 8 us), from 64 heads
// on the in-order issue of the unpipelined loop. Attention kernel, us, 128-head
// kernel -> this one: 1 x 512, 128 heads, fp16 16.2 -> 7.9 (kW = 8; 9.6 with
// 4); 1 x 8192, 128 heads 17.0 -> 11.6 (15.4 with 8); 32 x 4099 with 16 heads
// 51.3 -> 33.4, with 32 heads 52.2 -> 38.0; with 64 heads 52.7 -> 60.2 and 16
// queries over 2048 rows 21.7 -> 36.3 (both stay on the 128-head kernel: the
// plan's waves16). Two head blocks per workgroup (Q and O fill the registers)
// took 45.7 at 32 heads and 50.2 at 64.
#include "la_internal.hpp"

#include <hip/hip_ext.h>

namespace la {
namespace {

constexpr int kDc = 512;
constexpr int kDr = 64;
constexpr int kRowElems = kDc + kDr;
constexpr int kCtPitch = kDc * 2;       // 1024 B, chunks permuted by cf(row)
// fp32 queries taken in (kW = 8): 8-element slots of a row, and its 16-bit LDS
// pitch (73 16-B chunks: 16 rows at one chunk hit distinct banks)
constexpr int kSlots = kRowElems / 8;
constexpr int kQPitch = 2 * kRowElems + 16;

// Workgroup of kW waves, tile of 16 kW positions, 16 query heads.
template <int kW>
struct Lds {
  static constexpr int kT = 16 * kW;
  static constexpr int kRope = kT * kCtPitch;         // 128-B k_rope rows, chunks permuted by rf(row)
  static constexpr int kP = kRope + kT * 128;         // P: 16 heads x kT positions, 16-bit
  static constexpr int kPRow = 2 * kT;                // bytes per head
  static constexpr int kMax = kP + 16 * kPRow;        // kW wave maxima per head
  static constexpr int kBytes = kMax + 16 * 4 * kW;
  // epilogue: 16 heads x 512 fp16 at a 1040-B pitch, then per head the waves' row maxima and sums
  static constexpr int kStagePitch = 1040;
  static constexpr int kStat = 16 * kStagePitch;
  static_assert(kStat + 16 * 8 * kW <= kP, "epilogue staging fits the tile");
  static_assert(kW != 8 || kRope + 16 * kQPitch <= kBytes, "the queries fit the k_rope and P rows");
  static_assert((8 / kW) * kBytes <= 160 * 1024, "two waves per SIMD");
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) char lchar;

template <typename KT>
struct Ops16;
template <>
struct Ops16<__hip_bfloat16> {
  typedef bf16x8 vec;
  typedef __bf16 elem;
  static __device__ inline f32x4 mma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Ops16<__half> {
  typedef f16x8 vec;
  typedef _Float16 elem;
  static __device__ inline f32x4 mma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Chunk permutations: cf is one to one over 16 rows, and its upper three bits
// are over rows {0..3, 8..11} and over rows {4..7, 12..15} (the rows a half
// wave's transposed reads touch); rf is the 128-B-row swizzle.
__host__ __device__ constexpr int cf(int r) { return 2 * ((r & 3) | ((r & 8) >> 1)) | ((r >> 2) & 1); }
__host__ __device__ constexpr int rf(int r) { return (r >> 1) & 7; }
constexpr bool cf_ok() {
  unsigned all = 0, up[2] = {0, 0};
  for (int r = 0; r < 16; ++r) {
    all |= 1u << cf(r);
    up[(r >> 2) & 1] |= 1u << (cf(r) >> 1);
  }
  return all == 0xFFFF && up[0] == 0xFF && up[1] == 0xFF;
}
static_assert(cf_ok(), "bank spread of the c_t rows");

template <typename T>
__device__ inline T lds_ld(const lchar* L, int off) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(L + off);
}
template <typename T>
__device__ inline void lds_st(lchar* L, int off, T v) {
  *reinterpret_cast<__attribute__((address_space(3))) T*>(L + off) = v;
}
__device__ inline i16x4 lds_tr(const lchar* L, int off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(lds_void*)(L + off));
}

// max / sum of x over the four lanes l%16 + 16 g
__device__ inline float max_groups(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(u_of(x), u_of(x), false, false);
  x = fmaxf(f_of(r[0]), f_of(r[1]));
  r = __builtin_amdgcn_permlane16_swap(u_of(x), u_of(x), false, false);
  return fmaxf(f_of(r[0]), f_of(r[1]));
}
__device__ inline float sum_groups(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(u_of(x), u_of(x), false, false);
  x = f_of(r[0]) + f_of(r[1]);
  r = __builtin_amdgcn_permlane16_swap(u_of(x), u_of(x), false, false);
  return f_of(r[0]) + f_of(r[1]);
}

// KT: the MFMAs' type (bf16 for an FP8 cache). groups: workgroups per chunk.
// kW = 8 takes absorbed queries as they come (p.q_prep == nullptr): the
// workgroup scales and rounds its heads' rows as prep_q_kernel does and spreads
// them over its waves through LDS, under the first tile's copies. One launch
// less: 1 x 512 fp16 16.5 -> 14.8 us a call. (With every
// wave reading the fp32 rows itself, 32 B of a row per lane, the call was 4.7 us
// slower than with the launch.) kW = 4 has no room for it (its k_rope and P rows
// are smaller than the queries). zero_out (optional): zero_n floats zeroed for
// a half-row merge.
template <typename KT, int kW, bool kPaged, bool kFp8, bool kFilled>
__global__ __launch_bounds__(64 * kW, 2) void decode_mfma16_kernel(DecodeProblem p, int groups, float* zero_out,
                                                                  int zero_n) {
  typedef Ops16<KT> O_;
  typedef typename O_::vec vec;
  typedef typename O_::elem E;
  constexpr int kRowB = kFp8 ? kRowElems : 2 * kRowElems;
  typedef Lds<kW> D;
  typedef float fw __attribute__((ext_vector_type(kW)));
  constexpr int kT = D::kT;
  // P rows of 128 B swizzle like k_rope rows, rows of 256 B over all 16 heads
  constexpr auto pf = [](int r) { return kT == 128 ? r & 15 : rf(r); };
  constexpr int kCB = 32 / kW;   // 16-column blocks of O per wave
  static_assert(kCB <= 8, "a wave's value chunks lie in one permuted group of 16");
  constexpr int kKS = kT / 32;   // PV k-steps per tile
  constexpr int kAhead = 6;     // LDS operands in flight

  warm_kernarg_lines(p);
  extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
  lchar* L = (lchar*)lds_raw;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (zero_out)
    for (int i = blockIdx.x * 64 * kW + threadIdx.x; i < zero_n; i += gridDim.x * 64 * kW) zero_out[i] = 0.f;
  int chunk, group;
  block_coords(p.num_chunks, groups, &chunk, &group);
  if (chunk >= p.num_chunks) return;
  const int head0 = group * 16;  // Hq is a multiple of 16 (mfma_supported)

  ChunkWalk<kFilled> w;
  if (!walk_begin(p, chunk, group, w)) return;

  while (walk_next(p, w)) {
    const int s = w.s;
    const char* const seg_base = reinterpret_cast<const char*>(p.kv) + (kPaged ? 0 : (w.row0 + (w.lo - w.s_lo)) * kRowB);
    const uint32_t pos0 = (uint32_t)(w.lo - w.s_lo);
    const int last = (int)(w.seg_hi - w.lo - 1);
    const int ntiles = last / kT + 1;
    const int rlim = p.rope_rows > 0 ? (int)(p.rope_rows - 1) : INT32_MAX;

    // Q^T as the B operand: lane holds Q[head0 + n16][32kk + 8g .. +8], from
    // q_prep (in operand order, qprep_index), or from the fp32 queries' slots
    // (8 elements each) tid, tid + 512, tid + 1024, which go through LDS below
    vec q[18];
    const bool q32 = kW == 8 && !p.q_prep;
    f32x4 qf[kW == 8 ? 6 : 1];
    if (!q32) {
      const int ql = wave_lane();
      const int64_t qrow = (int64_t)s * qprep_rows_per_seq(p.Hq) + head0 + (ql & 15);
      const vec* qs =
          reinterpret_cast<const vec*>(reinterpret_cast<const E*>(p.q_prep) + qprep_index(qrow, 8 * (ql >> 4)));
#pragma unroll
      for (int kk = 0; kk < 18; ++kk) q[kk] = qs[128 * kk];
    }
    if constexpr (kW == 8) {
      if (q32) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const int slot = min((int)threadIdx.x + 512 * i, 16 * kSlots - 1);
          const int row = slot / kSlots, j = slot - row * kSlots;
          const int64_t hq = (int64_t)s * p.Hq + head0 + row;
          const float* src = j < kDc / 8 ? p.q_abs + hq * kDc + 8 * j : p.q_rope + hq * kDr + 8 * (j - kDc / 8);
          qf[2 * i] = reinterpret_cast<const f32x4*>(src)[0];
          qf[2 * i + 1] = reinterpret_cast<const f32x4*>(src)[1];
        }
      }
    }
    f32x4 o[kCB];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) o[cb] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = 0; t < ntiles; ++t) {
      // the tile's LDS addresses are made where they are used, from a fresh
      // lane index (held across the loop they would not fit beside Q and O)
      const int ln = wave_lane();
      // ---- stage the wave's 16 rows (rows past the segment re-read its last) ----
      const int pb = min(kT * t + 16 * wave, last);  // first row; the 16 lie in one block of a paged cache
      const int left = last - pb;
      const char* base;
      if constexpr (kPaged) {
        const uint32_t pos = pos0 + (uint32_t)pb, tile = pos >> 5;
        const uint32_t blk = (__umulhi(tile, p.tpb_magic) + tile) >> p.tpb_shift;
        const int e = min(max(p.block_table[(int64_t)s * p.blocks_per_seq + blk], 0), p.pool_last);
        const uint32_t row = (uint32_t)e * (uint32_t)p.block_size + (pos - blk * (uint32_t)p.block_size);
        base = reinterpret_cast<const char*>(p.kv) + (uint64_t)row * kRowB;
      } else {
        base = seg_base + (int64_t)pb * kRowB;
      }
      // k_rope: lane takes row lane/4, pairs 8 (lane%4) .. +7
      const int rr = ln >> 2, u = ln & 3;
      const int rrow = min(rr, left);
      const int rpos = min((int)pos0 + pb + rrow, rlim);
      const char* ksrc = base + rrow * kRowB + (kFp8 ? kDc : 2 * kDc);
      const f32x4* cs = reinterpret_cast<const f32x4*>(p.rope_cos + (int64_t)rpos * (kDr / 2) + 8 * u);
      const f32x4* sn = reinterpret_cast<const f32x4*>(p.rope_sin + (int64_t)rpos * (kDr / 2) + 8 * u);
      i16x8 ka, kb;
      u32x2 k8a, k8b;
      if constexpr (kFp8) {
        k8a = *reinterpret_cast<const u32x2*>(ksrc + 8 * u);
        k8b = *reinterpret_cast<const u32x2*>(ksrc + kDr / 2 + 8 * u);
      } else {
        ka = *reinterpret_cast<const i16x8*>(ksrc + 16 * u);
        kb = *reinterpret_cast<const i16x8*>(ksrc + kDr + 16 * u);
      }
      const f32x4 c0 = cs[0], c1 = cs[1], s0 = sn[0], s1 = sn[1];
      u32x2 x8[kFp8 ? 16 : 1];
      if (t > 0) lds_barrier();  // every wave is done with the previous tile
      if constexpr (kFp8) {
#pragma unroll
        for (int j = 0; j < 16; ++j) x8[j] = *reinterpret_cast<const u32x2*>(base + min(j, left) * kRowB + 8 * ln);
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j)
          __builtin_amdgcn_global_load_lds(base + (uint32_t)(min(j, left) * kRowB + 16 * (ln ^ cf(j))),
                                           (lds_void*)(L + (16 * wave + j) * kCtPitch), 16, 0, 0);
      }
      if constexpr (kW == 8) {
        if (q32 && t == 0) {  // the queries, in the place of the k_rope and P rows
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const int slot = (int)threadIdx.x + 512 * i;
            const int row = slot / kSlots, j = slot - row * kSlots;
            vec v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[e] = (E)(qf[2 * i][e] * p.scale_log2);
              v[4 + e] = (E)(qf[2 * i + 1][e] * p.scale_log2);
            }
            if (slot < 16 * kSlots) lds_st(L, D::kRope + row * kQPitch + 16 * j, v);
          }
          lds_barrier();
#pragma unroll
          for (int kk = 0; kk < 18; ++kk)
            q[kk] = lds_ld<vec>(L, D::kRope + (ln & 15) * kQPitch + 64 * kk + 16 * (ln >> 4));
          lds_barrier();
        }
      }
      {
        i16x8 ra, rb;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float k0, k1;
          if constexpr (kFp8) {
            const auto va = (e & 2) ? __builtin_amdgcn_cvt_pk_f32_fp8(k8a[e >> 2], true)
                                    : __builtin_amdgcn_cvt_pk_f32_fp8(k8a[e >> 2], false);
            const auto vb = (e & 2) ? __builtin_amdgcn_cvt_pk_f32_fp8(k8b[e >> 2], true)
                                    : __builtin_amdgcn_cvt_pk_f32_fp8(k8b[e >> 2], false);
            k0 = va[e & 1];
            k1 = vb[e & 1];
          } else {
            k0 = (float)__builtin_bit_cast(E, (short)ka[e]);
            k1 = (float)__builtin_bit_cast(E, (short)kb[e]);
          }
          const float c = e < 4 ? c0[e & 3] : c1[e & 3], sv = e < 4 ? s0[e & 3] : s1[e & 3];
          ra[e] = __builtin_bit_cast(short, (E)(k0 * c - k1 * sv));
          rb[e] = __builtin_bit_cast(short, (E)(k0 * sv + k1 * c));
        }
        const int row = D::kRope + (16 * wave + rr) * 128;
        lds_st(L, row + 16 * (u ^ rf(rr)), ra);
        lds_st(L, row + 16 * ((4 + u) ^ rf(rr)), rb);
      }
      if constexpr (kFp8) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          u32x4 y;
          y[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x8[j][0], 1.f, false));
          y[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x8[j][0], 1.f, true));
          y[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x8[j][1], 1.f, false));
          y[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x8[j][1], 1.f, true));
          lds_st(L, (16 * wave + j) * kCtPitch + 16 * (ln ^ cf(j)), y);
        }
      }
      // ---- scores of the wave's own rows: only its own copies have to land ----
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const int n16 = ln & 15, g = ln >> 4;
      const int row_l = 16 * wave + n16;
      const int ct0 = row_l * kCtPitch + 16 * (g ^ cf(n16));  // k-step 0; 64 (kk % 4) is an exclusive or
      f32x4 sc = {0.f, 0.f, 0.f, 0.f};
      // operands kAhead k-steps ahead (the scheduling barriers keep the compiler from reading all 18 at once)
      auto a_rd = [&](int kk) -> vec {
        return kk < 16 ? lds_ld<vec>(L, (ct0 ^ (64 * (kk & 3))) + 256 * (kk >> 2))
                       : lds_ld<vec>(L, (D::kRope + row_l * 128 + 16 * (g ^ rf(n16))) ^ (64 * (kk - 16)));
      };
      vec a[kAhead];
#pragma unroll
      for (int kk = 0; kk < kAhead; ++kk) a[kk] = a_rd(kk);
#pragma unroll
      for (int kk = 0; kk < 18; ++kk) {
        sc = O_::mma(a[kk % kAhead], q[kk], sc);
        if (kk + kAhead < 18) a[kk % kAhead] = a_rd(kk + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
      settle(sc);
      // lane: head n16, positions 16w + 4g + i
      const int valid = last + 1 - kT * t;
      if (valid < kT) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (16 * wave + 4 * g + i >= valid) sc[i] = -INFINITY;
      }
      const float mx = max_groups(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])));
      if (g == 0) lds_st(L, D::kMax + 4 * kW * n16 + 4 * wave, mx);
      lds_barrier();
      const fw wm = lds_ld<fw>(L, D::kMax + 4 * kW * n16);
      float m_new = m;
#pragma unroll
      for (int w = 0; w < kW; ++w) m_new = fmaxf(m_new, wm[w]);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      const bool moved = m_new != m;
      m = m_new;
      float sum = 0.f;
      i16x4 pk;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(sc[i] - m_new);
        sum += e;
        pk[i] = __builtin_bit_cast(short, (E)e);
      }
      l = l * alpha + sum;
      lds_st(L, D::kP + n16 * D::kPRow + 16 * ((2 * wave + (g >> 1)) ^ pf(n16)) + 8 * (g & 1), pk);
      if (t > 0 && __builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) o[cb] *= alpha;
      }
      lds_barrier();
      // ---- PV: O^T[column][head] += V^T[column][position] P^T[position][head] ----
      // value reads: rows 32ks + 8g + 4x + n16/4, columns 16 kCB w + 16cb + 4(n16%4)
      int tr[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int r = 8 * g + 4 * x + (n16 >> 2);
        tr[x] = r * kCtPitch + ((32 * kCB * wave + 8 * (n16 & 1)) ^ (16 * (((n16 >> 1) & 1) ^ cf(r & 15))));
      }
      vec pv[kKS];
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) pv[ks] = lds_ld<vec>(L, (D::kP + n16 * D::kPRow + 16 * (g ^ pf(n16))) ^ (64 * ks));
      auto v_rd = [&](int step) -> vec {
        const int off = 32 * kCtPitch * (step / kCB), cb = step % kCB;
        const i16x4 v0 = lds_tr(L, (tr[0] ^ (32 * cb)) + off);
        const i16x4 v1 = lds_tr(L, (tr[1] ^ (32 * cb)) + off);
        i16x8 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = v0[e];
          v[4 + e] = v1[e];
        }
        return __builtin_bit_cast(vec, v);
      };
      vec v[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) v[i] = v_rd(i);
#pragma unroll
      for (int i = 0; i < kKS * kCB; ++i) {
        o[i % kCB] = O_::mma(v[i % kAhead], pv[i / kCB], o[i % kCB]);
        if (i + kAhead < kKS * kCB) v[i % kAhead] = v_rd(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    // ---- segment end: the partial slot's rows, as decode_mfma_kernel writes them ----
    // fp16 N * 2^-e per half row, 2^(e-1) <= max |N| < 2^e; m and m + log2(l)
    lds_barrier();  // every wave is done with the tile
    const int lane = wave_lane();
    const int n16 = lane & 15, g = lane >> 4;
    const int64_t hq0 = (kFilled ? slot_of(p, chunk, s) : (int64_t)chunk + s) * p.Hq + head0;
    float rmax = 0.f;
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) settle(o[cb]);
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) rmax = fmaxf(rmax, fabsf(o[cb][i]));
    rmax = max_groups(rmax);
    l = sum_groups(l);
    if (g == 0) {
      lds_st(L, D::kStat + 8 * kW * n16 + 4 * wave, rmax);
      lds_st(L, D::kStat + 8 * kW * n16 + 4 * kW + 4 * wave, l);
    }
    lds_barrier();
    const fw rw = lds_ld<fw>(L, D::kStat + 8 * kW * n16), lw = lds_ld<fw>(L, D::kStat + 8 * kW * n16 + 4 * kW);
    const int half = wave / (kW / 2);  // this wave's half row
    float hmax = 0.f, lsum = 0.f;
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      if (w / (kW / 2) == half) hmax = fmaxf(hmax, rw[w]);
      lsum += lw[w];
    }
    const int ex = __builtin_amdgcn_frexp_expf(hmax);
    if (g == 0) {
      if (wave % (kW / 2) == 0) p.part_scale[2 * (hq0 + n16) + half] = __builtin_amdgcn_ldexpf(1.f, ex);
      if (wave == 0) {
        p.part_m[hq0 + n16] = m;
        p.part_lse[hq0 + n16] = m + log2f(lsum);
      }
    }
    const float mul = __builtin_amdgcn_ldexpf(1.f, -ex);
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      i16x4 h4;
#pragma unroll
      for (int i = 0; i < 4; ++i) h4[i] = __builtin_bit_cast(short, (_Float16)(o[cb][i] * mul));
      lds_st(L, n16 * D::kStagePitch + 32 * (kCB * wave + cb) + 8 * g, h4);
    }
    lds_barrier();
    char* const dst = reinterpret_cast<char*>(p.part_o) + hq0 * (kDc * 2) + 16 * lane;
#pragma unroll
    for (int j = 0; j < 16 / kW; ++j) {
      const int head = kW * j + wave;
      *reinterpret_cast<i16x8*>(dst + head * (kDc * 2)) = lds_ld<i16x8>(L, head * D::kStagePitch + 16 * lane);
    }
    lds_barrier();  // the staging is read before the next segment's tile lands on it
    w.lo = w.seg_hi;
    ++w.s;
  }
}

template <typename KT, int kW, bool kPaged, bool kFp8, bool kFilled>
hipError_t launch16_t(const DecodeProblem& p, hipStream_t stream, float* zero_out, int zero_n, hipEvent_t ev_begin,
                      hipEvent_t ev_end) {
  constexpr int lds = Lds<kW>::kBytes;
  static OncePerDevice once;
  const hipError_t e = allow_lds(once, reinterpret_cast<const void*>(&decode_mfma16_kernel<KT, kW, kPaged, kFp8, kFilled>), lds);
  if (e != hipSuccess) return e;
  const int groups = p.Hq / 16;
  const dim3 grid((unsigned)mfma_grid_blocks(p.num_chunks, groups));
  if (ev_begin || ev_end)
    hipExtLaunchKernelGGL((decode_mfma16_kernel<KT, kW, kPaged, kFp8, kFilled>), grid, dim3(64 * kW), lds, stream, ev_begin,
                          ev_end, 0, p, groups, zero_out, zero_n);
  else
    hipLaunchKernelGGL((decode_mfma16_kernel<KT, kW, kPaged, kFp8, kFilled>), grid, dim3(64 * kW), lds, stream, p, groups, zero_out,
                       zero_n);
  return hipGetLastError();
}

template <int kW, bool kPaged, bool kFilled>
hipError_t launch16_w(const DecodeProblem& p, hipStream_t stream, float* zero_out, int zero_n, hipEvent_t ev_begin,
                      hipEvent_t ev_end) {
  typedef __hip_bfloat16 B;
  if (p.kv_dtype == LA_DTYPE_FP8_E4M3)
    return launch16_t<B, kW, kPaged, true, kFilled>(p, stream, zero_out, zero_n, ev_begin, ev_end);
  if (p.kv_dtype == LA_DTYPE_BF16)
    return launch16_t<B, kW, kPaged, false, kFilled>(p, stream, zero_out, zero_n, ev_begin, ev_end);
  return launch16_t<__half, kW, kPaged, false, kFilled>(p, stream, zero_out, zero_n, ev_begin, ev_end);
}

template <int kW>
hipError_t launch16_k(const DecodeProblem& p, hipStream_t stream, float* zero_out, int zero_n, hipEvent_t ev_begin,
                      hipEvent_t ev_end) {
  if (p.block_table) return launch16_w<kW, true, true>(p, stream, zero_out, zero_n, ev_begin, ev_end);
  if (p.chunk_len < 0) return launch16_w<kW, false, true>(p, stream, zero_out, zero_n, ev_begin, ev_end);
  return launch16_w<kW, false, false>(p, stream, zero_out, zero_n, ev_begin, ev_end);
}

}  // namespace

hipError_t launch_decode_mfma16(const DecodeProblem& p, int waves, hipStream_t stream, float* zero_out, int64_t zero_n,
                                hipEvent_t ev_begin, hipEvent_t ev_end) {
  if (zero_n > INT32_MAX / 2) return hipErrorInvalidValue;  // the kernel counts in 32 bits
  return waves == 8 ? launch16_k<8>(p, stream, zero_out, (int)zero_n, ev_begin, ev_end)
                    : launch16_k<4>(p, stream, zero_out, (int)zero_n, ev_begin, ev_end);
}

}  // namespace la
