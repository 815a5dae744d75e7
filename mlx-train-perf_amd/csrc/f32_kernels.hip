// fp32 inputs: the fused linear cross-entropy and flash attention for fp32 hidden states / q, k, v
// (the reference kernels take fp32 as well as bf16: core/loss.py:24, attention/api.py:41-43).
//
// Arithmetic is fp32 end to end: fp32 MFMA products (exact fp32 multiplies, fp32 accumulation;
// v_mfma_f32_32x32x2_f32 in the LCE, v_mfma_f32_16x16x4_f32 in attention), fp32 softmax statistics,
// fp32 outputs and gradients. The algorithms are those of
// the bf16 kernels (lce_kernels.hip, attn_kernels.hip) and of the reference's oracles:
//   LCE forward: per token lse = logsumexp_v(h . w_v) (online over vocab tiles, vocab splits merged
//     by the finalize), tgt = h . w_y, nll = lse - tgt (core/naive.py:9-14, core/chunked.py:35-49);
//   LCE backward: g = (exp(z - lse) - onehot) * ct in fp32 per vocab chunk, dH = g . W_chunk,
//     dW = g^T . H (core/chunked.py:52-90);
//   attention: O = softmax(scale Q K^T + mask) V, L = row logsumexp; backward D = rowsum(dO O),
//     dS = P (dP - D), dQ = scale dS K, dK = scale dS^T Q, dV = P^T dO summed over each kv head's
//     query-head group (attention/reference.py:37-116, attention/api.py:126-194).
//
// MFMA 32x32x2 f32 lane layout (wave64): lane l supplies A[i = l % 32][k = l / 32] and
// B[k = l / 32][j = l % 32]; its 16 results are C[i = 8 (r / 4) + 4 (l / 32) + r % 4][j = l % 32]. Which k a
// lane half contracts at which step is each core's choice (both operands make the same), so that a lane
// reads consecutive k of its row: the register-staged core k = 8 h + s of 16, the copied one
// 8 c + 4 h + s of 32. The 16x16x4 layout stands at the attention kernels.
#include "mtp_common.hpp"
#include "mtp_launch.hpp"

namespace mtp {
namespace f32k {

__device__ __forceinline__ f32x16 mfma2(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void zero(f32x16& a) {
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = 0.f;
}
// Key (or query) index, within a 32-block, of accumulator register r of lane half h.
__device__ __forceinline__ int rrow(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// ------------------------------------------------------------------------------------------
// GEMM core: C[128][128] (+)= A[128][K] . B[128][K]^T over K in 16-deep LDS stages, 4 waves of
// 64 x 64 (wave w: A rows 64 (w & 1), B rows 64 (w >> 1)). Operand tiles are staged through
// registers into LDS in one of two layouts:
//   row: [128 rows][16 k] with a 20-float pitch (16-byte fragment reads of 16 lanes hit distinct
//        banks);
//   col: [16 k][128 rows] with a 132-float pitch (the two lane halves read disjoint banks).
// Sources: `RowSrc` (row-major [rows][ld], k along a row), `ColSrc` (k-major [k][ld], rows along a
// k row), and the 4-bit affine head in either role (`Q4RowSrc`, `Q4ColSrc`: w = s * q + b in fp32,
// 8 nibbles per u32, low first, scale and bias per 64 along the hidden dim). Out-of-range elements
// read as zero.
// ------------------------------------------------------------------------------------------
constexpr int kT = 128, kBK = 16, kRowPitch = 20, kColPitch = 132;
constexpr int kTileFloats = 2560;  // >= 128 * 20 and 16 * 132

struct RowSrc {
  static constexpr bool kCol = false;
  const float* p;
  long ld;
  int rows, K;
  bool vec;
  __device__ __forceinline__ float at(int r, int k) const { return (r < rows && k < K) ? p[(long)r * ld + k] : 0.f; }
  __device__ __forceinline__ f32x4 quad(int r, int k) const {
    if (vec && r < rows && k + 3 < K) return *reinterpret_cast<const f32x4*>(p + (long)r * ld + k);
    return f32x4{at(r, k), at(r, k + 1), at(r, k + 2), at(r, k + 3)};
  }
};
struct ColSrc {
  static constexpr bool kCol = true;
  const float* p;  // [k][ld], element (k, r)
  long ld;
  int rows, K;
  bool vec;
  __device__ __forceinline__ float at(int k, int r) const { return (r < rows && k < K) ? p[(long)k * ld + r] : 0.f; }
  __device__ __forceinline__ f32x4 quad(int k, int r) const {
    if (vec && k < K && r + 3 < rows) return *reinterpret_cast<const f32x4*>(p + (long)k * ld + r);
    return f32x4{at(k, r), at(k, r + 1), at(k, r + 2), at(k, r + 3)};
  }
};
// 4-bit head rows v (tile rows) along the hidden dim d (k): W[v][d].
struct Q4Geom {
  const uint32_t* wq;
  const float* sc;
  const float* bi;
  int D;
  __device__ __forceinline__ float w(long v, int d) const {
    const uint32_t word = wq[v * (D >> 3) + (d >> 3)];
    const long g = v * (D >> 6) + (d >> 6);
    return __builtin_fmaf(sc[g], (float)((word >> (4 * (d & 7))) & 0xFu), bi[g]);
  }
};
struct Q4RowSrc {
  static constexpr bool kCol = false;
  Q4Geom q;
  long v0;
  int rows, K;
  __device__ __forceinline__ f32x4 quad(int r, int k) const {
    f32x4 x;
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = (r < rows && k + u < K) ? q.w(v0 + r, k + u) : 0.f;
    return x;
  }
};
// The 4-bit head as the k-major operand: element (k = vocab row, r = hidden index).
struct Q4ColSrc {
  static constexpr bool kCol = true;
  Q4Geom q;
  long v0;
  int rows, K;  // rows: hidden dims from the tile start, K: vocab rows
  int d0;
  __device__ __forceinline__ f32x4 quad(int k, int r) const {
    f32x4 x;
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = (k < K && r + u < rows) ? q.w(v0 + k, d0 + r + u) : 0.f;
    return x;
  }
};

// One operand's share of a stage: thread t fetches quads idx = t + 256 p (p = 0, 1) of the 512.
template <class Src>
__device__ __forceinline__ void fetch(const Src& s, int k0, f32x4 (&x)[2]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int idx = t + 256 * p;
    if constexpr (Src::kCol) x[p] = s.quad(k0 + (idx >> 5), 4 * (idx & 31));
    else x[p] = s.quad(idx >> 2, k0 + 4 * (idx & 3));
  }
}
template <bool COL>
__device__ __forceinline__ void put(const f32x4 (&x)[2], float* lds) {
  const int t = threadIdx.x;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int idx = t + 256 * p;
    const int off = COL ? (idx >> 5) * kColPitch + 4 * (idx & 31) : (idx >> 2) * kRowPitch + 4 * (idx & 3);
    *reinterpret_cast<f32x4*>(lds + off) = x[p];
  }
}
// Fragments of the wave's two 32-row blocks for the 8 steps of a stage: v[b][s].
template <bool COL>
__device__ __forceinline__ void frags(const float* lds, int r0, float (&v)[2][8]) {
  const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    if constexpr (COL) {
#pragma unroll
      for (int s = 0; s < 8; ++s) v[b][s] = lds[(8 * h + s) * kColPitch + r0 + 32 * b + i];
    } else {
      const float* row = lds + (r0 + 32 * b + i) * kRowPitch + 8 * h;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(row);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(row + 4);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        v[b][s] = lo[s];
        v[b][4 + s] = hi[s];
      }
    }
  }
}

// acc[bi][bj] = C[64 (w & 1) + 32 bi + ..][64 (w >> 1) + 32 bj + ..]. `lds` holds 4 tiles:
// [stage][A, B].
template <class SA, class SB>
__device__ __forceinline__ void gemm128(const SA& sa, const SB& sb, int K, float* lds, f32x16 (&acc)[2][2]) {
  const int w = threadIdx.x >> 6;
  const int ra = 64 * (w & 1), rb = 64 * (w >> 1);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) zero(acc[i][j]);
  const int nk = (K + kBK - 1) / kBK;
  f32x4 xa[2], xb[2];
  fetch(sa, 0, xa);
  fetch(sb, 0, xb);
  put<SA::kCol>(xa, lds);
  put<SB::kCol>(xb, lds + kTileFloats);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    float* cur = lds + (kt & 1) * 2 * kTileFloats;
    float* nxt = lds + ((kt + 1) & 1) * 2 * kTileFloats;
    if (kt + 1 < nk) {
      fetch(sa, (kt + 1) * kBK, xa);
      fetch(sb, (kt + 1) * kBK, xb);
    }
    float fa[2][8], fb[2][8];
    frags<SA::kCol>(cur, ra, fa);
    frags<SB::kCol>(cur + kTileFloats, rb, fb);
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma2(fa[i][s], fb[j][s], acc[i][j]);
    if (kt + 1 < nk) {
      put<SA::kCol>(xa, nxt);
      put<SB::kCol>(xb, nxt + kTileFloats);
    }
    __syncthreads();
  }
}

// The waves' copies have landed and their LDS reads are done, for the whole workgroup.
__device__ __forceinline__ void copies_landed() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
}
// One global -> LDS copy of a wave: 16 (4) bytes per lane from src + voff (lanes past `bytes` get zeros)
// to dst + 16 lane (4 lane), dst wave-uniform.
__device__ __forceinline__ void lds_copy16(const float* src, int bytes, char* dst, uint32_t voff) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), (short)0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, 0, 0, 0);
}
__device__ __forceinline__ void lds_copy4(const float* src, int bytes, char* dst, uint32_t voff) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), (short)0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, voff, 0, 0, 0);
}

// ------------------------------------------------------------------------------------------
// The same product on copied tiles (dense operands whose rows are multiples of 16 bytes): 32-deep stages of
// 16 KiB per operand, copied global -> LDS one stage ahead, one barrier per stage; two workgroups per CU.
// The matrix pipe bounds it (4096 MFMA cycles per wave and stage against 32 KiB copied and 16 KiB
// read); the register-staged core above stalls on its loads and LDS writes. N = 1024, D = 512, V = 32000, the
// kernels' times in one trace: forward 363 -> 305 us, gradient tiles 391 -> 343, dH 367 -> 302; the whole
// step 1043 -> 827 us (122 of the 153 TFLOP/s a library fp32 matrix product reaches). Two 256-register
// waves per SIMD: left to a budget of 512 the compiler moved the accumulators between VGPRs and AGPRs
// in every stage.
//   RowOp: k along a row: [128 rows][32 k], chunk c (4 k) of row r at slot c ^ swz32(r); a lane reads chunk
//          2 c + h of its row for the 4 steps of c.
//   ColOp: k-major: [32 k][128 columns]; a lane reads columns 2 i and 2 i + 1 of the k rows of its half, so
//          block b of a wave holds the columns 2 i + b.
// Lane half h contracts k = 8 c + 4 h + s at step s of c, in both. Rows, k and columns past the end read
// as zeros or (columns of a k-major operand) as neighbours whose results are not stored.
// ------------------------------------------------------------------------------------------
constexpr int kDK = 32, kOpB = 16384;
__device__ __forceinline__ int swz32(int r) { return (r ^ ((r >> 3) & 3)) & 7; }
__device__ __forceinline__ int range31(long bytes) { return bytes <= 0 ? 0 : bytes > 0x7fffffffL ? 0x7fffffff : (int)bytes; }

struct RowOp {
  const float* p;  // tile row 0, k = 0
  long ld;
  int rows, K;     // rows from the tile start, contraction length
  uint32_t voff;   // this lane's offset in its wave's copy 0; copy m lies 32 m rows on
  int ck;          // first k of the lane's chunk
  __device__ __forceinline__ RowOp(const float* p_, long ld_, int rows_, int K_) : p(p_), ld(ld_), rows(rows_ < kT ? rows_ : kT), K(K_) {
    const int lane = threadIdx.x & 63, row = 8 * (threadIdx.x >> 6) + (lane >> 3);
    ck = 4 * ((lane & 7) ^ swz32(row));
    voff = 4u * (uint32_t)(row * (int)ld + ck);
  }
  static __device__ __forceinline__ int pos(int b, int i) { return 32 * b + i; }
  __device__ __forceinline__ void copy(int kt, char* dst) const {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), left = K - kt * kDK;
    // (a gradient tile's row may end inside a chunk: its zeros up to the chunk's end are read too)
    const int bytes = left > 0 ? range31(4 * ((rows - 1) * ld + ((left + 3) & ~3))) : 0;
    const uint32_t v = ck < left ? voff : 0x60000000u;  // past the end of its row: nothing
#pragma unroll
    for (int m = 0; m < 4; ++m) lds_copy16(p + kt * kDK, bytes, dst + 1024 * (4 * m + w), v + 128u * m * (uint32_t)ld);
  }
  __device__ __forceinline__ void frags(const char* st, int first, int c, float (&v)[2][4]) const {
    const int i = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1, row = first + i;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(st + row * 128 + (((h ^ swz32(row)) << 4) ^ (c << 5)) + 4096 * b);
#pragma unroll
      for (int s = 0; s < 4; ++s) v[b][s] = x[s];
    }
  }
};
struct ColOp {
  const float* p;  // k = 0, tile column 0
  long ld;
  int cols, K;     // columns from the tile start to the end of the row, contraction length
  uint32_t voff;   // this lane's offset in its wave's copy 0; copy m lies 8 m k rows on
  __device__ __forceinline__ ColOp(const float* p_, long ld_, int cols_, int K_) : p(p_), ld(ld_), cols(cols_), K(K_) {
    const int lane = threadIdx.x & 63;
    voff = 4u * (uint32_t)((2 * (threadIdx.x >> 6) + (lane >> 5)) * (int)ld + 4 * (lane & 31));
  }
  static __device__ __forceinline__ int pos(int b, int i) { return 2 * i + b; }
  __device__ __forceinline__ void copy(int kt, char* dst) const {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), left = K - kt * kDK;
    const int bytes = left > 0 ? range31(4 * ((left - 1) * ld + cols)) : 0;
#pragma unroll
    for (int m = 0; m < 4; ++m) lds_copy16(p + kt * kDK * ld, bytes, dst + 1024 * (4 * m + w), voff + 32u * m * (uint32_t)ld);
  }
  __device__ __forceinline__ void frags(const char* st, int first, int c, float (&v)[2][4]) const {
    const int i = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const f32x2 x = *reinterpret_cast<const f32x2*>(st + (8 * c + 4 * h + s) * 512 + 4 * (first + 2 * i));
      v[0][s] = x[0];
      v[1][s] = x[1];
    }
  }
};
// acc[bi][bj] = C[64 (w & 1) + OA::pos(bi, ..)][64 (w >> 1) + OB::pos(bj, ..)]; s0 and s1 hold A, then B.
template <class OA, class OB>
__device__ __forceinline__ void gemm128_copied(const OA& oa, const OB& ob, int K, char* s0, char* s1, f32x16 (&acc)[2][2]) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ra = 64 * (w & 1), rb = 64 * (w >> 1);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) zero(acc[i][j]);
  const int nk = (K + kDK - 1) / kDK;
  auto stage = [&](int kt, const char* cur, char* nxt) __attribute__((always_inline)) {
    oa.copy(kt + 1, nxt);  // past the end: nothing read, zeros into a stage nobody reads
    ob.copy(kt + 1, nxt + kOpB);
    float fa[2][2][4], fb[2][2][4];  // one chunk pair ahead
    oa.frags(cur, ra, 0, fa[0]);
    ob.frags(cur + kOpB, rb, 0, fb[0]);
    // Keeps the copies up here (the scheduler sank the last one to its wait) and each chunk pair's
    // reads ahead of the products they run under.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c < 3) {
        oa.frags(cur, ra, c + 1, fa[(c + 1) & 1]);
        ob.frags(cur + kOpB, rb, c + 1, fb[(c + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma2(fa[c & 1][i][s], fb[c & 1][j][s], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    copies_landed();
  };
  oa.copy(0, s0);
  ob.copy(0, s0 + kOpB);
  copies_landed();
  for (int kt = 0; kt < nk; kt += 2) {
    stage(kt, s0, s1);
    if (kt + 1 < nk) stage(kt + 1, s1, s0);
  }
}

__device__ __forceinline__ bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }
// Head kinds of the kernels below: dense (any hidden dim), 4-bit, dense on the copied-tile core.
constexpr int kDense = 0, kQ4 = 1, kCopied = 2;
template <int KIND>
constexpr int kStage0 = KIND == kCopied ? 2 * kOpB : 4 * kTileFloats * 4;
template <int KIND>
constexpr int kStage1 = KIND == kCopied ? 2 * kOpB : 16;

// ------------------------------------------------------------------------------------------
// LCE forward: workgroup (128-token tile, vocab split) walks the split's 128-column vocab tiles;
// C[v][t] = W_v . H_t, so each lane owns token columns and keeps an online (max, sum of exp2) per
// token, merged with lane ^ 32 and the other vocab-half wave at the end into part_m/part_s
// [split][N] (log2 domain), which the finalize merges.
// ------------------------------------------------------------------------------------------
template <int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lce32_fwd_kernel(const float* __restrict__ H, const float* __restrict__ W,
                                                        const uint32_t* __restrict__ Wq, const float* __restrict__ Sc,
                                                        const float* __restrict__ Bi, int N, int D, int V, int nsplit,
                                                        float* __restrict__ part_m, float* __restrict__ part_s) {
  __shared__ __attribute__((aligned(1024))) char s0[kStage0<KIND>];
  __shared__ __attribute__((aligned(1024))) char s1[kStage1<KIND>];
  float* lds = reinterpret_cast<float*>(s0);
  const int t0 = blockIdx.x * kT, split = blockIdx.y;
  const int vtiles = (V + kT - 1) / kT;
  const int per = (vtiles + nsplit - 1) / nsplit;
  const int vt0 = split * per, vt1 = (vt0 + per < vtiles) ? vt0 + per : vtiles;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wa = w & 1, wb = w >> 1, h = lane >> 5;
  RowSrc hb{H + (long)t0 * D, D, N - t0, D, aligned16(H) && D % 4 == 0};
  float m[2] = {kNegInf, kNegInf}, s[2] = {0.f, 0.f};
  for (int vt = vt0; vt < vt1; ++vt) {
    const int v0 = vt * kT;
    f32x16 acc[2][2];
    if constexpr (KIND == kCopied) {
      gemm128_copied(RowOp(W + (long)v0 * D, D, V - v0, D), RowOp(H + (long)t0 * D, D, N - t0, D), D, s0, s1, acc);
    } else if constexpr (KIND == kQ4) {
      Q4RowSrc wa_{Q4Geom{Wq, Sc, Bi, D}, v0, V - v0, D};
      gemm128(wa_, hb, D, lds, acc);
    } else {
      RowSrc wa_{W + (long)v0 * D, D, V - v0, D, aligned16(W) && D % 4 == 0};
      gemm128(wa_, hb, D, lds, acc);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float mz = kNegInf;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int v = v0 + 64 * wa + 32 * i + rrow(r, h);
          if (v >= V) acc[i][j][r] = kNegInf;
          mz = fmaxf(mz, acc[i][j][r]);
        }
      const float mn = fmaxf(m[j], mz * kLog2e);
      const float base = (mn == kNegInf) ? 0.f : mn;
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += fast_exp2(__builtin_fmaf(acc[i][j][r], kLog2e, -base));
      s[j] = s[j] * fast_exp2(m[j] - base) + sum;
      m[j] = mn;
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) lse2_merge(m[j], s[j], __shfl_xor(m[j], 32, 64), __shfl_xor(s[j], 32, 64));
  __syncthreads();
  float* xm = lds;
  float* xs = lds + 128;
  if (wa == 1 && h == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      xm[64 * wb + 32 * j + (lane & 31)] = m[j];
      xs[64 * wb + 32 * j + (lane & 31)] = s[j];
    }
  }
  __syncthreads();
  if (wa == 0 && h == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int tl = 64 * wb + 32 * j + (lane & 31);
      lse2_merge(m[j], s[j], xm[tl], xs[tl]);
      if (t0 + tl < N) {
        part_m[(long)split * N + t0 + tl] = m[j];
        part_s[(long)split * N + t0 + tl] = s[j];
      }
    }
  }
}

// Per token (one wave each): merge the splits into lse, tgt = H_t . W_y as an fp32 dot product,
// ignore_index rows nll = 0 and tgt = 0, out-of-range targets tgt = 0 (nll = lse).
template <int Q4>
__global__ __launch_bounds__(256) void lce32_finalize_kernel(const float* __restrict__ H, const float* __restrict__ W,
                                                             const uint32_t* __restrict__ Wq, const float* __restrict__ Sc,
                                                             const float* __restrict__ Bi, const int64_t* __restrict__ targets,
                                                             int N, int D, int V, int nsplit, const float* __restrict__ part_m,
                                                             const float* __restrict__ part_s, long long ignore_index,
                                                             float* __restrict__ nll, float* __restrict__ lse,
                                                             float* __restrict__ tgt) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= N) return;
  float mm = kNegInf, ss = 0.f;
  for (int sp = lane; sp < nsplit; sp += 64) lse2_merge(mm, ss, part_m[(long)sp * N + t], part_s[(long)sp * N + t]);
  const float gm = wave_max(mm);
  const float base = (gm == kNegInf) ? 0.f : gm;
  const float gs = wave_sum(ss * fast_exp2(mm - base));
  const float l = (base + fast_log2(gs)) * kLn2;
  const long long y = targets[t];
  const bool ignored = y == ignore_index;
  const bool inrange = y >= 0 && y < (long long)V;
  float dot = 0.f;
  if (!ignored && inrange) {
    const float* h = H + (long)t * D;
    if constexpr (Q4) {
      const Q4Geom q{Wq, Sc, Bi, D};
      for (int d = lane; d < D; d += 64) dot = __builtin_fmaf(h[d], q.w(y, d), dot);
    } else {
      const float* wr = W + (long)y * D;
      for (int d = lane; d < D; d += 64) dot = __builtin_fmaf(h[d], wr[d], dot);
    }
    dot = wave_sum(dot);
  }
  if (lane == 0) {
    lse[t] = l;
    tgt[t] = (ignored || !inrange) ? 0.f : dot;
    nll[t] = ignored ? 0.f : l - ((!inrange) ? 0.f : dot);
  }
}

// Gradient tile of the backward: C[t][v] = H_t . W_v for rows [row0, row0 + nrows) and the chunk's
// columns [c0, c0 + ncols); G[t][v - c0] = (exp(C - lse_t) - [v == y_t]) * coef_t in fp32, coef_t =
// d_nll[t] (0 for ignored rows), 0 past the vocab end (up to a multiple of 4 columns, which the dH
// product reads).
template <int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lce32_bwd_g_kernel(const float* __restrict__ H, const float* __restrict__ W,
                                                          const uint32_t* __restrict__ Wq, const float* __restrict__ Sc,
                                                          const float* __restrict__ Bi, const int64_t* __restrict__ targets,
                                                          const float* __restrict__ lse, const float* __restrict__ dnll,
                                                          int D, int V, long long ignore_index, int row0, int nrows,
                                                          int c0, int ncols, float* __restrict__ G, long ldg) {
  __shared__ __attribute__((aligned(1024))) char s0[kStage0<KIND>];
  __shared__ __attribute__((aligned(1024))) char s1[kStage1<KIND>];
  float* lds = reinterpret_cast<float*>(s0);
  const int tt = blockIdx.x * kT, vv = blockIdx.y * kT;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wa = w & 1, wb = w >> 1, h = lane >> 5;
  RowSrc hs{H + (long)(row0 + tt) * D, D, nrows - tt, D, aligned16(H) && D % 4 == 0};
  const int v0 = c0 + vv;
  // Per row: coefficient, log2-domain lse and the target's column in the chunk (-1: none), fetched ahead
  // of the product (it has barriers between these writes and the reads below).
  __shared__ float rcoef[kT], rl2[kT];
  __shared__ int ry[kT];
  if (threadIdx.x < kT) {
    const int t = row0 + tt + threadIdx.x;
    const bool ok = tt + (int)threadIdx.x < nrows;
    const long long y = ok ? targets[t] : -1;
    rcoef[threadIdx.x] = ok && y != ignore_index ? dnll[t] : 0.f;
    rl2[threadIdx.x] = ok ? lse[t] * kLog2e : 0.f;
    ry[threadIdx.x] = y >= c0 && y - c0 < ncols ? (int)(y - c0) : -1;
  }
  f32x16 acc[2][2];
  if constexpr (KIND == kCopied) {
    gemm128_copied(RowOp(H + (long)(row0 + tt) * D, D, nrows - tt, D), RowOp(W + (long)v0 * D, D, V - v0, D), D, s0, s1, acc);
  } else if constexpr (KIND == kQ4) {
    Q4RowSrc ws{Q4Geom{Wq, Sc, Bi, D}, v0, V - v0, D};
    gemm128(hs, ws, D, lds, acc);
  } else {
    RowSrc ws{W + (long)v0 * D, D, V - v0, D, aligned16(W) && D % 4 == 0};
    gemm128(hs, ws, D, lds, acc);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rl = 64 * wa + 32 * i + rrow(r, h), tl = tt + rl;
      if (tl >= nrows) continue;
      const float coef = rcoef[rl], l2 = rl2[rl];
      const int y = ry[rl];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int vl = vv + 64 * wb + 32 * j + (lane & 31);
        if (vl >= ((ncols + 3) & ~3)) continue;
        float g = 0.f;
        if (c0 + vl < V) {
          const float p = fast_exp2(__builtin_fmaf(acc[i][j][r], kLog2e, -l2));
          g = (p - (vl == y ? 1.f : 0.f)) * coef;
        }
        G[(long)tl * ldg + vl] = g;
      }
    }
}

// Stores (ACC: adds) a product's tile to C[M][N]: blockIdx.x: 128 rows, blockIdx.y: 128 columns. PA, PB: the
// operands' order of rows within a wave's 64 (the register-staged sources have RowOp's).
template <bool ACC, class PA = RowOp, class PB = RowOp>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[2][2], int M, int N, float* __restrict__ C, long ldc) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wa = w & 1, wb = w >> 1, h = lane >> 5;
  const int m0 = blockIdx.x * kT, n0 = blockIdx.y * kT;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + 64 * wa + PA::pos(i, rrow(r, h));
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + 64 * wb + PB::pos(j, lane & 31);
        if (n >= N) continue;
        float* c = C + (long)m * ldc + n;
        *c = ACC ? *c + acc[i][j][r] : acc[i][j][r];
      }
    }
}

// dH[t][d] (+)= sum_v G[t][v] W[v][d] over one chunk: A = G rows, B = the chunk's W rows read k-major.
// dH for one vocab chunk, its contraction (the chunk's columns) split into parts of `per` columns
// (blockIdx.z = part; one part: per >= kcols) so that a small output grid still fills the GPU. With
// one part the tile goes to dH (written by the first chunk, accumulated by the others); with several,
// each part's tile goes to its own fp32 slice part_out[z] and lce32_dh_reduce_kernel sums them in
// part order.
template <int KIND, bool ACC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lce32_dh_kernel(const float* __restrict__ G, long ldg, const float* __restrict__ W,
                                                       const uint32_t* __restrict__ Wq, const float* __restrict__ Sc,
                                                       const float* __restrict__ Bi, int D, int c0, int kcols, int per,
                                                       int nrows, float* __restrict__ dH) {
  __shared__ __attribute__((aligned(1024))) char s0[kStage0<KIND>];
  __shared__ __attribute__((aligned(1024))) char s1[kStage1<KIND>];
  float* lds = reinterpret_cast<float*>(s0);
  const int m0 = blockIdx.x * kT, n0 = blockIdx.y * kT;
  const int k0 = blockIdx.z * per;
  const int kn = (kcols - k0 < per) ? kcols - k0 : per;
  float* out = dH + (long)blockIdx.z * nrows * D;
  f32x16 acc[2][2];
  if constexpr (KIND == kCopied) {
    gemm128_copied(RowOp(G + (long)m0 * ldg + k0, ldg, nrows - m0, kn), ColOp(W + (long)(c0 + k0) * D + n0, D, D - n0, kn),
                   kn, s0, s1, acc);
    store_tile<ACC, RowOp, ColOp>(acc, nrows, D, out, D);
  } else {
    RowSrc ga{G + (long)m0 * ldg + k0, ldg, nrows - m0, kn, ldg % 4 == 0};
    if constexpr (KIND == kQ4) {
      Q4ColSrc wb{Q4Geom{Wq, Sc, Bi, D}, (long)c0 + k0, D - n0, kn, n0};
      gemm128(ga, wb, kn, lds, acc);
    } else {
      ColSrc wb{W + (long)(c0 + k0) * D + n0, D, D - n0, kn, aligned16(W) && D % 4 == 0};
      gemm128(ga, wb, kn, lds, acc);
    }
    store_tile<ACC>(acc, nrows, D, out, D);
  }
}

// dH (+)= sum over p of parts[p], in part order (deterministic), over the n x d elements.
template <bool ACC>
__global__ __launch_bounds__(256) void lce32_dh_reduce_kernel(const float* __restrict__ parts, int nparts, long count,
                                                              float* __restrict__ dH) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float x = ACC ? dH[i] : 0.f;
  for (int p = 0; p < nparts; ++p) x += parts[(long)p * count + i];
  dH[i] = x;
}

// dW[v][d] = sum_t G[t][v] H[t][d] for one chunk's vocab rows (all tokens): A = G read k-major
// (k = t), B = H read k-major.
template <int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lce32_dw_kernel(const float* __restrict__ G, long ldg, const float* __restrict__ H,
                                                       int N, int D, int vrows, float* __restrict__ dW) {
  __shared__ __attribute__((aligned(1024))) char s0[kStage0<KIND>];
  __shared__ __attribute__((aligned(1024))) char s1[kStage1<KIND>];
  const int m0 = blockIdx.x * kT, n0 = blockIdx.y * kT;
  f32x16 acc[2][2];
  if constexpr (KIND == kCopied) {
    gemm128_copied(ColOp(G + m0, ldg, (int)ldg - m0, N), ColOp(H + n0, D, D - n0, N), N, s0, s1, acc);
    store_tile<false, ColOp, ColOp>(acc, vrows, D, dW, D);
  } else {
    ColSrc ga{G + m0, ldg, vrows - m0, N, ldg % 4 == 0};
    ColSrc hb{H + n0, D, D - n0, N, aligned16(H) && D % 4 == 0};
    gemm128(ga, hb, N, reinterpret_cast<float*>(s0), acc);
    store_tile<false>(acc, vrows, D, dW, D);
  }
}

// ------------------------------------------------------------------------------------------
// Attention on v_mfma_f32_16x16x4_f32 (lane l: col = l % 16, g = l / 16; it supplies A[col][g] and
// B[g][col] and holds C[4 g + r][col], r < 4). A wave owns 16 positions of one head as the MFMA columns
// (queries: forward and dQ; keys: dK/dV) and keeps their rows and gradients in registers; the 8 waves
// of a workgroup share 32-position tiles of the other side, copied global -> LDS one tile ahead.
//
// The matrix pipe bounds it: a 16x16x4 product takes 32 cycles of its SIMD, so a forward tile is 4096
// MFMA cycles per wave against 32 KiB of LDS reads and ~100 VALU instructions. 32-position waves on
// tiles staged through registers between two barriers left most of it idle: at S = 2048 (16/4 heads,
// head_dim 128, causal) one wave per SIMD waited at the barriers, and the 64 key blocks of dK/dV, of very
// unequal work, were all that 256 CUs had. Hence 16-position waves, which need half the registers, and
// a workgroup of two half-workgroups of 4 waves on two position blocks: under the causal mask the
// mirrored pair (block p and block n - 1 - p), whose work adds up to the same for every pair, with one
// wave of each on every SIMD; otherwise two adjacent blocks, which read the same tiles.
// Measured there: forward 456 -> 177 us, dQ 570 -> 242, dK/dV 2537 -> 322 (4 splits and their sum), 97-109
// TFLOP/s; at S = 8192, 32/8 heads 4.08, 6.19 and 8.13 ms, 133-135 of the 153 TFLOP/s a library fp32
// matrix product reaches.
//
// Row reads (products over head_dim): lane (col, g) reads 16-byte chunks of row col, chunk order
// row_chunk(c, g) -- the contraction may visit head_dim in any order as long as both operands do.
// Column reads (products over the tile's positions): lane (col, g) reads chunk 16 b + col of row
// 4 g + s, one read for four products, whose output rows are head_dims 64 b + 4 i + j (product j, row
// i). Chunk k of row r sits at slot k ^ (r % 16): the 16 lanes of a g, and the lanes 0-7 / 32-39 of a
// read, fall on distinct banks in both.
//
// Masks: key j visible to query i iff j < S, (causal) j <= i, (packed) seg_start[i] <= j; in the
// packed layout (contiguous, ascending, gapless segments) that is "same segment and j <= i".
// ------------------------------------------------------------------------------------------
constexpr int kPos = 32;  // positions per LDS tile

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <int DH>
struct ALay {
  static constexpr int kRowB = DH == 64 ? 256 : 512;  // 96: chunks 24-31 of a row stay empty (zeros)
  static constexpr int kTile = kPos * kRowB;
  static constexpr int kSlots = kRowB / 16;           // lanes per row of a 1 KiB copy
  static constexpr int kM = kTile / 8192;             // copies per wave and tile
  static constexpr int kC = DH / 16;                  // chunks per lane and row
  static constexpr int kB = DH / 16;                  // 16-row accumulator blocks over head_dim
};

// The per-lane constants of a wave.
template <int DH>
struct ALane {
  using L = ALay<DH>;
  int col, g;
  int rb, rt;            // row-read byte offsets: chunks 0-15 (rb) and, head_dim 96, 16-23 (rt), row `col`
  int cb, ct;            // column-read byte offsets of row 4 g at s = 0
  uint32_t src[L::kM];   // global byte offsets of this lane's copies, from the tile's first row
  __device__ __forceinline__ void init() {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    col = lane & 15;
    g = lane >> 4;
    rb = col * L::kRowB + (((8 * (g >> 1) + (g & 1)) ^ col) << 4);
    rt = col * L::kRowB + (((4 * (g >> 1) + (g & 1)) ^ col) << 4) + 256;
    cb = 4 * g * L::kRowB + ((col ^ (4 * g)) << 4);
    ct = 4 * g * L::kRowB + (((col >> 1) ^ (4 * g)) << 4) + 8 * (col & 1) + 256;
#pragma unroll
    for (int m = 0; m < L::kM; ++m) {
      const int row = (64 / L::kSlots) * (w + 8 * m) + lane / L::kSlots;
      const int c = (lane % L::kSlots) ^ (row & 15);
      src[m] = 16 * c < 4 * DH ? (uint32_t)(row * 4 * DH + 16 * c) : 0x7ffffff0u;  // past the range: zeros
    }
  }
  // Byte offset within a global row of the lane's chunk c.
  __device__ __forceinline__ int row_chunk(int c) const {
    if (DH == 96 && c >= 4) return 16 * (16 + 4 * (g >> 1) + 2 * (c - 4) + (g & 1));
    return 16 * (16 * (c >> 2) + 8 * (g >> 1) + 2 * (c & 3) + (g & 1));
  }
  // Chunk c of tile row 16 half + col.
  __device__ __forceinline__ f32x4 row(const char* tile, int half, int c) const {
    const int off = (DH == 96 && c >= 4) ? (rt ^ ((c - 4) << 5)) : (rb ^ ((c & 3) << 5)) + ((c >> 2) << 8);
    return *reinterpret_cast<const f32x4*>(tile + off + 16 * half * L::kRowB);
  }
  // Four head_dims 64 b + 4 col + j (j < 4) of tile row 16 half + 4 g + s.
  __device__ __forceinline__ f32x4 cols(const char* tile, int half, int s, int b) const {
    return *reinterpret_cast<const f32x4*>(tile + (cb ^ (s << 4)) + (16 * half + s) * L::kRowB + (b << 8));
  }
  // head_dim 96: the last 32, 64 + 2 col + j (j < 2).
  __device__ __forceinline__ f32x2 cols_tail(const char* tile, int half, int s) const {
    return *reinterpret_cast<const f32x2*>(tile + (ct ^ (s << 4)) + (16 * half + s) * L::kRowB);
  }
  // This wave's copies of the 32 rows from position p0 of a [S][DH] matrix (rows past S as zeros;
  // nothing read, zeros written, when not live).
  __device__ __forceinline__ void copy(const float* m, int p0, int S, char* tile, bool live) const {
    const int rows = S - p0 < kPos ? S - p0 : kPos;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < L::kM; ++i)
      lds_copy16(m + (live ? (long)p0 * DH : 0), live ? rows * 4 * DH : 0, tile + 1024 * (w + 8 * i), src[i]);
  }
  // The lane's chunks of a global row as the B operand of the head_dim products.
  __device__ __forceinline__ void load_row(const float* row, bool valid, f32x4 (&x)[L::kC]) const {
#pragma unroll
    for (int c = 0; c < L::kC; ++c) {
      x[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (valid) x[c] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(row) + row_chunk(c));
    }
  }
  // acc[half] = tile rows . x (head_dim contraction), the two 16-row chains interleaved.
  __device__ __forceinline__ void dot_rows(const char* tile, const f32x4 (&x)[L::kC], f32x4 (&acc)[2]) const {
    acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < L::kC; ++c) {
      const f32x4 a = row(tile, 0, c), b = row(tile, 1, c);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        acc[0] = mfma4(a[s], x[c][s], acc[0]);
        acc[1] = mfma4(b[s], x[c][s], acc[1]);
      }
    }
  }
  // out += tile^T . p over the tile's 32 rows, p[half][r] the weight of row 16 half + 4 g + r.
  __device__ __forceinline__ void dot_cols(const char* tile, const f32x4 (&p)[2], f32x4 (&out)[L::kB]) const {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int b = 0; b < DH / 64; ++b) {
          const f32x4 a = cols(tile, half, s, b);
#pragma unroll
          for (int j = 0; j < 4; ++j) out[4 * b + j] = mfma4(a[j], p[half][s], out[4 * b + j]);
        }
        if constexpr (DH == 96) {
          const f32x2 a = cols_tail(tile, half, s);
          out[4] = mfma4(a[0], p[half][s], out[4]);
          out[5] = mfma4(a[1], p[half][s], out[5]);
        }
      }
  }
  // Writes acc (head_dim x this lane's position) * mul to the position's global row.
  __device__ __forceinline__ void store_row(float* row, const f32x4 (&acc)[L::kB], float mul) const {
#pragma unroll
    for (int b = 0; b < DH / 64; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f32x4*>(row + 64 * b + 16 * g + 4 * r) =
            f32x4{acc[4 * b][r] * mul, acc[4 * b + 1][r] * mul, acc[4 * b + 2][r] * mul, acc[4 * b + 3][r] * mul};
    if constexpr (DH == 96) {
#pragma unroll
      for (int r = 0; r < 4; r += 2)
        *reinterpret_cast<f32x4*>(row + 64 + 8 * g + 2 * r) =
            f32x4{acc[4][r] * mul, acc[5][r] * mul, acc[4][r + 1] * mul, acc[5][r + 1] * mul};
    }
  }
};
// Sum and maximum over the four lanes (g = 0..3) of a column.
__device__ __forceinline__ float col_sum(float x) {
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}
__device__ __forceinline__ float col_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16, 64));
  return fmaxf(x, __shfl_xor(x, 32, 64));
}
// The two position blocks of pair p out of n: mirrored (the causal mask: equal work per pair) or
// adjacent. The second may be n (none).
__host__ __device__ __forceinline__ void pair_blocks(int p, int n, bool mirror, int& a, int& b) {
  a = mirror ? p : 2 * p;
  b = mirror ? n - 1 - p : 2 * p + 1;
  if (b <= a) b = n;
}
__host__ __device__ __forceinline__ int q_heads32(int G) { return G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1; }

// Forward (DQ = false) and dQ (DQ = true). A half-workgroup holds q_heads32(G) heads of one GQA group x
// 16 (4 / heads) queries: every K/V tile feeds all of them.
template <int DH, bool PACKED, bool DQ>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(DQ ? 2 : 4)))
void attn32_q_kernel(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                     const float* __restrict__ d_o, const float* __restrict__ o_in, const float* __restrict__ lse_in,
                     float* __restrict__ dvec, const int32_t* __restrict__ seg_start, float* __restrict__ out,
                     float* __restrict__ lse_out, int B, int Hq, int Hkv, int S, float scale, int causal) {
  using L = ALay<DH>;
  __shared__ __attribute__((aligned(1024))) char lds0[2 * L::kTile];  // K, V
  __shared__ __attribute__((aligned(1024))) char lds1[2 * L::kTile];
  const int G = Hq / Hkv, hpw = q_heads32(G), R = 16 * (4 / hpw);
  const int nqb = (S + R - 1) / R, hgb = Hq / hpw, nhg = B * hgb;
  const int hg = blockIdx.x % nhg, b = hg / hgb, h0 = (hg % hgb) * hpw, kvh = h0 / G;
  int pa, pb;
  pair_blocks((int)(blockIdx.x / nhg), nqb, causal && !PACKED, pa, pb);
  ALane<DH> ln;
  ln.init();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = w & 3;
  const int blk = w < 4 ? pa : pb;
  const int head = h0 + u % hpw, qw0 = blk * R + 16 * (u / hpw), qi = qw0 + ln.col;
  const bool wave_has = blk < nqb && qw0 < S, qvalid = wave_has && qi < S;
  const int wq_last = qw0 + 15 < S ? qw0 + 15 : S - 1;
  const long qrow = (long)(b * Hq + head) * S;
  const float* kh = k + (long)(b * Hkv + kvh) * S * DH;
  const float* vh = v + (long)(b * Hkv + kvh) * S * DH;
  const int32_t* sst = PACKED ? seg_start + (long)b * S : nullptr;
  const float scale_log2 = scale * kLog2e;

  f32x4 qx[L::kC], dx[DQ ? L::kC : 1];
  ln.load_row(q + (qrow + qi) * DH, qvalid, qx);
  float l2q = 0.f, dq_row = 0.f;
  if constexpr (DQ) {
    ln.load_row(d_o + (qrow + qi) * DH, qvalid, dx);
    f32x4 ox[L::kC];
    ln.load_row(o_in + (qrow + qi) * DH, qvalid, ox);
    float dp = 0.f;
#pragma unroll
    for (int c = 0; c < L::kC; ++c)
#pragma unroll
      for (int s = 0; s < 4; ++s) dp = __builtin_fmaf(dx[c][s], ox[c][s], dp);
    dq_row = col_sum(dp);
    if (qvalid && ln.g == 0) dvec[qrow + qi] = dq_row;
    l2q = qvalid ? lse_in[qrow + qi] * kLog2e : 0.f;
  }
  // Keys of the workgroup: those of its last block (the latest queries) and, packed, from its first
  // block's first segment on (adjacent blocks: one contiguous range).
  const int last = pb < nqb ? pb : pa;
  const int kv_end = (causal && (last + 1) * R < S) ? (last + 1) * R : S;
  const int kv_begin = PACKED ? (sst[pa * R] / kPos) * kPos : 0;
  const int ntiles = (kv_end - kv_begin + kPos - 1) / kPos;
  const int my_sst = (PACKED && qvalid) ? sst[qi] : 0;
  const int w_sst_first = (PACKED && wave_has) ? __builtin_amdgcn_readfirstlane(sst[qw0]) : 0;
  const int w_sst_last = (PACKED && wave_has) ? __builtin_amdgcn_readfirstlane(sst[wq_last]) : 0;

  float m = kNegInf, l = 0.f;
  f32x4 acc[L::kB];
#pragma unroll
  for (int i = 0; i < L::kB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  ln.copy(kh, kv_begin, S, lds0, ntiles > 0);  // no tile (a segment start past the queries): nothing read
  ln.copy(vh, kv_begin, S, lds0 + L::kTile, ntiles > 0);
  copies_landed();
  // The row loads are complete here: tell the compiler, which would wait for them (and for the copies
  // in flight) at their first use.
#pragma unroll
  for (int c = 0; c < L::kC; ++c) {
    asm volatile("" : "+v"(qx[c]));
    if constexpr (DQ) asm volatile("" : "+v"(dx[c]));
  }

  auto body = [&](int t, const char* cur, char* nxt) __attribute__((always_inline)) {
    const int kv0 = kv_begin + t * kPos;
    ln.copy(kh, kv0 + kPos, S, nxt, t + 1 < ntiles);
    ln.copy(vh, kv0 + kPos, S, nxt + L::kTile, t + 1 < ntiles);
    if (wave_has && !(causal && kv0 > wq_last) && !(PACKED && kv0 + kPos - 1 < w_sst_first)) {
      f32x4 sc[2];
      ln.dot_rows(cur, qx, sc);  // S^T = K Q^T
      // Only tiles across the wave's diagonal, the sequence end or a segment start hold hidden pairs.
      const bool need_mask = (causal && kv0 + kPos - 1 > qw0) || kv0 + kPos > S || (PACKED && kv0 < w_sst_last);
      const int hi = (causal ? (qi < S - 1 ? qi : S - 1) : S - 1) - kv0 - 4 * ln.g, lo = my_sst - kv0 - 4 * ln.g;
      auto visible = [&](int half, int r) { return 16 * half + r <= hi && (!PACKED || 16 * half + r >= lo); };
      if constexpr (DQ) {
        f32x4 dp[2];
        ln.dot_rows(cur + L::kTile, dx, dp);  // dP^T = V dO^T
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[half][r] = fast_exp2(__builtin_fmaf(sc[half][r], scale_log2, -l2q));
        if (need_mask) {
#pragma unroll
          for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[half][r] = visible(half, r) ? sc[half][r] : 0.f;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[half][r] *= dp[half][r] - dq_row;
        ln.dot_cols(cur, sc, acc);  // dQ^T += K^T dS^T
      } else {
        float mx = kNegInf;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[half][r] *= scale_log2;
        if (need_mask) {
#pragma unroll
          for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[half][r] = visible(half, r) ? sc[half][r] : kNegInf;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, fmaxf(sc[0][r], sc[1][r]));
        const float mn = fmaxf(m, col_max(mx));
        const float base = (mn == kNegInf) ? 0.f : mn;
        // O and l are rescaled when some query's maximum rose; alpha is 1 for the others.
        if (__builtin_amdgcn_ballot_w64(mn > m) != 0) {
          const float alpha = fast_exp2(m - base);  // m = -inf: 0 (O and l are 0)
          l *= alpha;
#pragma unroll
          for (int i = 0; i < L::kB; ++i) acc[i] *= alpha;
          m = mn;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            sc[half][r] = fast_exp2(sc[half][r] - base);
            l += sc[half][r];
          }
        ln.dot_cols(cur + L::kTile, sc, acc);  // O^T += V^T P^T
      }
    }
    copies_landed();
  };
  for (int t = 0; t < ntiles; t += 2) {
    body(t, lds0, lds1);
    if (t + 1 < ntiles) body(t + 1, lds1, lds0);
  }
  if constexpr (DQ) {
    if (qvalid) ln.store_row(out + (qrow + qi) * DH, acc, scale);
  } else {
    const float lt = col_sum(l);
    if (!qvalid) return;
    if (ln.g == 0) lse_out[qrow + qi] = (lt > 0.f) ? (m + fast_log2(lt)) * kLn2 : kNegInf;
    ln.store_row(out + (qrow + qi) * DH, acc, lt > 0.f ? 1.f / lt : 0.f);
  }
}

// dK, dV: a half-workgroup holds a block of 64 keys of one kv head, each wave 16 of them with their K
// and V rows; items (query head h of the group, 32-query tile t) visit the queries that see the pair of
// blocks. They are dealt to nsplit workgroups, item (h, t) to (h + t) % nsplit (attn32_dkv_splits), so
// that a key's partial sums do not depend on the block it is paired with (one packed segment gives the
// causal result bit for bit); with several, each writes an fp32 partial
// part[split][dK | dV][b][kv head][key][d], which attn32_dkv_reduce_kernel sums in split order.
template <int DH, bool PACKED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void attn32_dkv_kernel(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                       const float* __restrict__ d_o, const float* __restrict__ lse, const float* __restrict__ dvec,
                       const int32_t* __restrict__ seg_start, float* __restrict__ dk, float* __restrict__ dv, int B,
                       int Hq, int Hkv, int S, float scale, int causal, int nsplit, float* __restrict__ part) {
  using L = ALay<DH>;
  __shared__ __attribute__((aligned(1024))) char lds0[2 * L::kTile + 512];  // Q, dO, L (32 of 64), D (32 of 64)
  __shared__ __attribute__((aligned(1024))) char lds1[2 * L::kTile + 512];
  const int G = Hq / Hkv, nkb = (S + 63) / 64, nbh = B * Hkv;
  const int split = blockIdx.x % nsplit, bh = (blockIdx.x / nsplit) % nbh, b = bh / Hkv, kvh = bh % Hkv;
  int ba, bb;
  pair_blocks((int)(blockIdx.x / nsplit / nbh), nkb, causal && !PACKED, ba, bb);
  ALane<DH> ln;
  ln.init();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = w < 4 ? ba : bb, kw0 = blk * 64 + 16 * (w & 3), kj = kw0 + ln.col;
  const bool wave_has = blk < nkb && kw0 < S, kvalid = wave_has && kj < S;
  const long krow = (long)bh * S;
  const float scale_log2 = scale * kLog2e;
  const int32_t* sst = PACKED ? seg_start + (long)b * S : nullptr;

  f32x4 kx[L::kC], vx[L::kC];
  ln.load_row(k + (krow + kj) * DH, kvalid, kx);
  ln.load_row(v + (krow + kj) * DH, kvalid, vx);
  // Query tiles [t0, t1) see the workgroup's keys; queries q < my_lim see key kj (packed: those of its
  // segment), and the wave's keys none from w_end on.
  const int t0 = causal ? ba * (64 / kPos) : 0;
  int t1 = (S + kPos - 1) / kPos, my_lim = S, w_lim = S, w_end = S;
  if (PACKED) {
    auto above = [&](int x) {  // the end of position x's segment
      int lo = x, hi = S;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sst[mid] > x) hi = mid;
        else lo = mid + 1;
      }
      return lo;
    };
    const int last = bb < nkb ? bb : ba, wl = kw0 + 15 < S ? kw0 + 15 : S - 1;
    t1 = (__builtin_amdgcn_readfirstlane(above(last * 64 + 63 < S ? last * 64 + 63 : S - 1)) + kPos - 1) / kPos;
    if (kvalid) my_lim = above(kj);
    w_lim = __builtin_amdgcn_readfirstlane(my_lim);  // the first key's: the smallest
    if (wave_has) w_end = __builtin_amdgcn_readfirstlane(above(wl));
  }
  struct Item {
    int h, t;
  };
  auto settle = [&](Item x) __attribute__((always_inline)) {  // the first item of this split from x on (h = G: none)
    while (x.h < G && x.t >= t1) {
      ++x.h;
      int r = (split - x.h - t0) % nsplit;
      if (r < 0) r += nsplit;
      x.t = t0 + r;
    }
    return x;
  };

  f32x4 dka[L::kB], dva[L::kB];
#pragma unroll
  for (int i = 0; i < L::kB; ++i) dka[i] = dva[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Copies of an item into a stage: Q and dO rows, L and D (waves 0 and 1, 32 floats each).
  auto copy = [&](Item x, char* st) __attribute__((always_inline)) {
    const bool live = x.h < G;
    const int q0 = x.t * kPos;
    const long qrow = (long)(b * Hq + kvh * G + (live ? x.h : 0)) * S;
    ln.copy(q + qrow * DH, q0, S, st, live);
    ln.copy(d_o + qrow * DH, q0, S, st + L::kTile, live);
    if (w < 2) {
      const int rows = S - q0 < kPos ? S - q0 : kPos;
      lds_copy4((w ? dvec : lse) + qrow + (live ? q0 : 0), live ? rows * 4 : 0, st + 2 * L::kTile + 256 * w,
                  4u * (threadIdx.x & 63));
    }
  };
  auto body = [&](Item x, Item next, const char* cur, char* nxt) __attribute__((always_inline)) {
    copy(next, nxt);
    const int q0 = x.t * kPos;
    if (wave_has && !(causal && q0 + kPos - 1 < kw0) && !(PACKED && q0 >= w_end)) {
      f32x4 p[2], ds[2];
      ln.dot_rows(cur, kx, p);              // S = Q K^T (queries x this lane's key)
      ln.dot_rows(cur + L::kTile, vx, ds);  // dP = dO V^T
      const float* sl = reinterpret_cast<const float*>(cur + 2 * L::kTile);
      const bool need_mask = (causal && q0 < kw0 + 15) || q0 + kPos > S || (PACKED && q0 + kPos > w_lim);
      const int lo = causal ? kj - q0 - 4 * ln.g : -kPos, hi = my_lim - q0 - 4 * ln.g;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(sl + 16 * half + 4 * ln.g);
#pragma unroll
        for (int r = 0; r < 4; ++r) p[half][r] = fast_exp2(__builtin_fmaf(p[half][r], scale_log2, -l4[r] * kLog2e));
      }
      if (need_mask) {
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < 4; ++r) p[half][r] = (16 * half + r >= lo && 16 * half + r < hi) ? p[half][r] : 0.f;
      }
      ln.dot_cols(cur + L::kTile, p, dva);  // dV^T += dO^T P
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(sl + 64 + 16 * half + 4 * ln.g);
#pragma unroll
        for (int r = 0; r < 4; ++r) ds[half][r] = p[half][r] * (ds[half][r] - d4[r]);
      }
      ln.dot_cols(cur, ds, dka);  // dK^T += Q^T dS
    }
    copies_landed();
  };
  Item x = settle(Item{-1, t1});
  if (x.h < G) {
    copy(x, lds0);
    copies_landed();
#pragma unroll
    for (int c = 0; c < L::kC; ++c) asm volatile("" : "+v"(kx[c]), "+v"(vx[c]));
    while (true) {
      const Item y = settle(Item{x.h, x.t + nsplit});
      body(x, y, lds0, lds1);
      if (y.h >= G) break;
      x = settle(Item{y.h, y.t + nsplit});
      body(y, x, lds1, lds0);
      if (x.h >= G) break;
    }
  }
  if (!kvalid) return;
  const long plane = (long)nbh * S * DH;
  if (nsplit > 1) {
    dk = part + 2L * split * plane;
    dv = dk + plane;
  }
  ln.store_row(dk + (krow + kj) * DH, dka, scale);
  ln.store_row(dv + (krow + kj) * DH, dva, 1.f);
}

// dK (blockIdx.y 0) or dV (1) = the sum of the nsplit partials in split order. plane: floats, a multiple of 4.
__global__ __launch_bounds__(256) void attn32_dkv_reduce_kernel(const float* __restrict__ part, int nsplit, long plane,
                                                                float* __restrict__ dk, float* __restrict__ dv) {
  const long e = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (e >= plane) return;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  for (int sp = 0; sp < nsplit; ++sp) x += *reinterpret_cast<const f32x4*>(part + (2L * sp + blockIdx.y) * plane + e);
  *reinterpret_cast<f32x4*>((blockIdx.y ? dv : dk) + e) = x;
}

}  // namespace f32k

// ------------------------------------------------------------------------------------------
// Launchers
// ------------------------------------------------------------------------------------------
using namespace f32k;

// Vocab splits of the fp32 forward: about two workgroups per CU.
int lce32_fwd_nsplit(long N, long V) {
  const long rt = (N + kT - 1) / kT, vt = (V + kT - 1) / kT;
  long ns = (2L * kNumCU + rt - 1) / rt;
  if (ns > vt) ns = vt;
  if (ns > 1024) ns = 1024;
  return ns < 1 ? 1 : (int)ns;
}

// The copied-tile core takes dense operands whose rows start at multiples of 16 bytes (the entry points
// check the bases) and whose 128-row tiles stay below the 31-bit offsets of a copy.
static bool copied_tiles(long d, long ld) { return d % 4 == 0 && ld % 4 == 0 && d < (1L << 21) && ld < (1L << 21); }

hipError_t launch_lce32_fwd(const LceHead32& h, const float* H, const int64_t* targets, int N, int D, int V,
                            long long ignore_index, float* nll, float* lse, float* tgt, float* ws, hipStream_t st) {
  const int ns = lce32_fwd_nsplit(N, V);
  float* pm = ws;
  float* ps = ws + (long)ns * N;
  dim3 grid((N + kT - 1) / kT, ns), block(256);
  if (h.q4) hipLaunchKernelGGL(lce32_fwd_kernel<kQ4>, grid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, N, D, V, ns, pm, ps);
  else if (copied_tiles(D, D)) hipLaunchKernelGGL(lce32_fwd_kernel<kCopied>, grid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, N, D, V, ns, pm, ps);
  else hipLaunchKernelGGL(lce32_fwd_kernel<kDense>, grid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, N, D, V, ns, pm, ps);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  dim3 fgrid((N + 3) / 4);
  if (h.q4) hipLaunchKernelGGL(lce32_finalize_kernel<1>, fgrid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, targets, N, D, V, ns, pm, ps, ignore_index, nll, lse, tgt);
  else hipLaunchKernelGGL(lce32_finalize_kernel<0>, fgrid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, targets, N, D, V, ns, pm, ps, ignore_index, nll, lse, tgt);
  return hipGetLastError();
}

// Contraction parts of the fp32 dH product of a chunk of kcols columns: about two workgroups per
// CU over the ceil(N/128) x ceil(D/128) output tiles, each part at least 512 columns (32 stages of the
// register-staged core, 16 of the copied one) and a multiple of 16 (the copied core reads zeros past a
// part's end); at most 32. *per receives the columns per part.
int lce32_dh_parts(long N, long D, long kcols, int* per) {
  const long tiles = ((N + kT - 1) / kT) * ((D + kT - 1) / kT);
  long np = (2L * kNumCU + tiles - 1) / tiles;
  if (np > kcols / 512) np = kcols / 512;
  if (np > 32) np = 32;
  if (np < 1) np = 1;
  long pc = (kcols + np - 1) / np;
  pc = (pc + kBK - 1) / kBK * kBK;
  np = (kcols + pc - 1) / pc;
  if (per) *per = (int)(np == 1 ? kcols : pc);
  return (int)np;
}

hipError_t launch_lce32_bwd(const LceHead32& h, const float* H, const int64_t* targets, const float* lse,
                            const float* dnll, int N, int D, int V, long long ignore_index, int chunk, float* dH,
                            float* dW, float* Gbuf, hipStream_t st) {
  const long ldg = (long)chunk + 4;
  const bool copied = copied_tiles(D, ldg);
  dim3 block(256);
  for (int c0 = 0; c0 < V; c0 += chunk) {
    const int kc = (V - c0 < chunk) ? V - c0 : chunk;
    dim3 ggrid((N + kT - 1) / kT, (kc + kT - 1) / kT);
    if (h.q4) hipLaunchKernelGGL(lce32_bwd_g_kernel<kQ4>, ggrid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, targets, lse, dnll, D, V, ignore_index, 0, N, c0, kc, Gbuf, ldg);
    else if (copied) hipLaunchKernelGGL(lce32_bwd_g_kernel<kCopied>, ggrid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, targets, lse, dnll, D, V, ignore_index, 0, N, c0, kc, Gbuf, ldg);
    else hipLaunchKernelGGL(lce32_bwd_g_kernel<kDense>, ggrid, block, 0, st, H, h.w, h.wq, h.sc, h.bi, targets, lse, dnll, D, V, ignore_index, 0, N, c0, kc, Gbuf, ldg);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const bool acc = c0 > 0;
    int per = kc;
    const int np = lce32_dh_parts(N, D, kc, &per);
    dim3 hgrid((N + kT - 1) / kT, (D + kT - 1) / kT, np);
    if (np == 1) {
      if (h.q4) {
        if (acc) hipLaunchKernelGGL((lce32_dh_kernel<kQ4, true>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
        else hipLaunchKernelGGL((lce32_dh_kernel<kQ4, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
      } else if (copied) {
        if (acc) hipLaunchKernelGGL((lce32_dh_kernel<kCopied, true>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
        else hipLaunchKernelGGL((lce32_dh_kernel<kCopied, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
      } else {
        if (acc) hipLaunchKernelGGL((lce32_dh_kernel<kDense, true>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
        else hipLaunchKernelGGL((lce32_dh_kernel<kDense, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, dH);
      }
    } else {
      float* parts = Gbuf + (long)N * ldg;   // after the gradient tile: [np][N][D]
      if (h.q4) hipLaunchKernelGGL((lce32_dh_kernel<kQ4, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, parts);
      else if (copied) hipLaunchKernelGGL((lce32_dh_kernel<kCopied, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, parts);
      else hipLaunchKernelGGL((lce32_dh_kernel<kDense, false>), hgrid, block, 0, st, Gbuf, ldg, h.w, h.wq, h.sc, h.bi, D, c0, kc, per, N, parts);
      e = hipGetLastError();
      if (e != hipSuccess) return e;
      const long count = (long)N * D;
      dim3 rgrid((unsigned)((count + 255) / 256));
      if (acc) hipLaunchKernelGGL(lce32_dh_reduce_kernel<true>, rgrid, block, 0, st, parts, np, count, dH);
      else hipLaunchKernelGGL(lce32_dh_reduce_kernel<false>, rgrid, block, 0, st, parts, np, count, dH);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (dW) {
      dim3 wgrid((kc + kT - 1) / kT, (D + kT - 1) / kT);
      if (copied) hipLaunchKernelGGL(lce32_dw_kernel<kCopied>, wgrid, block, 0, st, Gbuf, ldg, H, N, D, kc, dW + (long)c0 * D);
      else hipLaunchKernelGGL(lce32_dw_kernel<kDense>, wgrid, block, 0, st, Gbuf, ldg, H, N, D, kc, dW + (long)c0 * D);
      e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

// Splits of each pair of key blocks in the fp32 dK/dV pass. One 8-wave workgroup per CU: the count that
// takes the fewest rounds x items (an item, 32 queries of one head against a pair: about 7 us) plus
// the partials' write and read (28 MB in the time of an item).
int attn32_dkv_splits(int b, int hq, int hkv, int s, int dh) {
  if (b < 1 || hkv < 1 || s < 1 || hq % hkv) return 1;
  const long pairs = ((s + 63) / 64 + 1) / 2, wgs = pairs * b * hkv, items = (long)(hq / hkv) * ((s + kPos - 1) / kPos);
  const long plane = (long)b * hkv * s * dh * 4;
  auto cost = [&](long ns) { return (wgs * ns + kNumCU - 1) / kNumCU * ((items + ns - 1) / ns) * 28000000L + (ns > 1 ? 4 * ns * plane : 0); };
  int best = 1;
  for (int ns = 2; ns <= 16 && ns <= items; ++ns)
    if (cost(ns) < cost(best)) best = ns;
  return best;
}
// D, then, from the next 256-byte boundary, the partials of a split dK/dV pass.
size_t attn32_bwd_workspace(int b, int hq, int hkv, int s, int dh, int ns) {
  return (size_t)b * hq * s * sizeof(float) + (ns > 1 ? 256 + (size_t)ns * 2 * b * hkv * s * dh * sizeof(float) : 0);
}

namespace {
dim3 grid32_q(const AttnShape& sh) {
  const int hpw = q_heads32(sh.hq / sh.hkv), R = 16 * (4 / hpw);
  return dim3(((sh.s + R - 1) / R + 1) / 2 * sh.b * (sh.hq / hpw));
}
template <int DH>
hipError_t fwd32_dh(const AttnShape& sh, const float* q, const float* k, const float* v, const int32_t* sst, float* o,
                    float* lse, hipStream_t st) {
  const dim3 grid = grid32_q(sh), block(512);
  if (sst) hipLaunchKernelGGL((attn32_q_kernel<DH, true, false>), grid, block, 0, st, q, k, v, nullptr, nullptr, nullptr, nullptr, sst, o, lse, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal);
  else hipLaunchKernelGGL((attn32_q_kernel<DH, false, false>), grid, block, 0, st, q, k, v, nullptr, nullptr, nullptr, nullptr, sst, o, lse, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal);
  return hipGetLastError();
}
template <int DH>
hipError_t bwd32_dh(const AttnShape& sh, const float* q, const float* k, const float* v, const float* o,
                    const float* lse, const float* d_o, const int32_t* sst, float* dq, float* dk, float* dv,
                    float* dvec, int ns, hipStream_t st) {
  const dim3 qgrid = grid32_q(sh), block(512);
  if (sst) hipLaunchKernelGGL((attn32_q_kernel<DH, true, true>), qgrid, block, 0, st, q, k, v, d_o, o, lse, dvec, sst, dq, nullptr, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal);
  else hipLaunchKernelGGL((attn32_q_kernel<DH, false, true>), qgrid, block, 0, st, q, k, v, d_o, o, lse, dvec, sst, dq, nullptr, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  float* part = reinterpret_cast<float*>(((uintptr_t)(dvec + (size_t)sh.b * sh.hq * sh.s) + 255) / 256 * 256);
  const dim3 kgrid(((sh.s + 63) / 64 + 1) / 2 * sh.b * sh.hkv * ns);
  if (sst) hipLaunchKernelGGL((attn32_dkv_kernel<DH, true>), kgrid, block, 0, st, q, k, v, d_o, lse, dvec, sst, dk, dv, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal, ns, part);
  else hipLaunchKernelGGL((attn32_dkv_kernel<DH, false>), kgrid, block, 0, st, q, k, v, d_o, lse, dvec, sst, dk, dv, sh.b, sh.hq, sh.hkv, sh.s, sh.scale, sh.causal, ns, part);
  e = hipGetLastError();
  if (e != hipSuccess || ns == 1) return e;
  const long plane = (long)sh.b * sh.hkv * sh.s * DH;
  hipLaunchKernelGGL(attn32_dkv_reduce_kernel, dim3((unsigned)((plane / 4 + 255) / 256), 2), dim3(256), 0, st, part, ns, plane, dk, dv);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_attn32_fwd(const AttnShape& sh, const float* q, const float* k, const float* v,
                             const int32_t* seg_start, float* o, float* lse, hipStream_t st) {
  switch (sh.dh) {
    case 64: return fwd32_dh<64>(sh, q, k, v, seg_start, o, lse, st);
    case 96: return fwd32_dh<96>(sh, q, k, v, seg_start, o, lse, st);
    case 128: return fwd32_dh<128>(sh, q, k, v, seg_start, o, lse, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_attn32_bwd(const AttnShape& sh, const float* q, const float* k, const float* v, const float* o,
                             const float* lse, const float* d_o, const int32_t* seg_start, float* dq, float* dk,
                             float* dv, float* dvec, int nsplit, hipStream_t st) {
  switch (sh.dh) {
    case 64: return bwd32_dh<64>(sh, q, k, v, o, lse, d_o, seg_start, dq, dk, dv, dvec, nsplit, st);
    case 96: return bwd32_dh<96>(sh, q, k, v, o, lse, d_o, seg_start, dq, dk, dv, dvec, nsplit, st);
    case 128: return bwd32_dh<128>(sh, q, k, v, o, lse, d_o, seg_start, dq, dk, dv, dvec, nsplit, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mtp
