// GEMM on 16-bit matrices (binary16 / bfloat16): C = alpha * op(A) * op(B) + beta * C with fp32
// accumulation on v_mfma_f32_32x32x16_{f16,bf16} and one rounding at the store -- the Linear layers of
// a half model (the reference calls cublasHgemm: src/core/tensor/tensor_math_cuda.h:1163-1187).
//
// A workgroup of four wavefronts owns a 64 x 64 tile of C, a wavefront a 32 x 32 quarter.  Both matrix
// operands want, per lane, eight consecutive reduction indices of one tile row, so both LDS tiles are
// [row][k] with k contiguous (pitch 32 + 8 halves: 16-byte reads without bank conflicts).  How a tile is
// staged depends on which index is contiguous in memory: with k contiguous (A not transposed, B
// transposed) a thread copies one octet with a 16-byte load; with the row index contiguous (A transposed,
// B not transposed) it loads eight rows of one k with a 16-byte load and writes them as eight 2-byte LDS
// stores; pointers, pitches or edges that do not allow the 16-byte access fall back to single elements.
// This kernel does not split the reduction.  Problems with few output tiles take the second kernel of this file, which splits it
// over the wavefronts of a workgroup and adds their sums in a fixed order: results are run-to-run identical either way.
#include <hip/hip_runtime.h>

#include "common.h"
#include "storage.h"

namespace {

constexpr int GT = 256, GBM = 64, GBN = 64, GBK = 32, GPITCH = GBK + 8;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <bool BF16>
__device__ __forceinline__ f32x16 mfma16(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

struct Operand {
  const uint16_t *p;
  int ld;        // row pitch of the stored matrix, in elements
  int k_contig;  // 1: element (row, k) at p[row * ld + k]; 0: at p[k * ld + row]
  int vec_ok;    // pointer and pitch allow 16-byte accesses
  int rows;      // rows of op(matrix): M for A, N for B
};

// Stages rows [row0, row0 + 64) x reduction indices [k0, k0 + 32) of `o` into tile[row][k]; what lies
// outside the matrix is written as zero.
__device__ __forceinline__ void stage(const Operand &o, int row0, int k0, int K, uint16_t *tile) {
  const int t = threadIdx.x;
  if (o.k_contig) {
    const int r = t >> 2, kk = (t & 3) * 8;   // one octet of k per thread
    const int row = row0 + r, k = k0 + kk;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < o.rows && k < K) {
      const uint16_t *src = o.p + size_t(row) * o.ld + k;
      if (o.vec_ok && k + 8 <= K) {
        v = *reinterpret_cast<const u32x4 *>(src);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k + j < K) v[j >> 1] |= unsigned(src[j]) << (16 * (j & 1));
      }
    }
    *reinterpret_cast<u32x4 *>(tile + r * GPITCH + kk) = v;
  } else {
    const int kk = t >> 3, rr = (t & 7) * 8;  // eight rows of one k per thread
    const int k = k0 + kk, row = row0 + rr;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (k < K && row < o.rows) {
      const uint16_t *src = o.p + size_t(k) * o.ld + row;
      if (o.vec_ok && row + 8 <= o.rows) {
        v = *reinterpret_cast<const u32x4 *>(src);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (row + j < o.rows) v[j >> 1] |= unsigned(src[j]) << (16 * (j & 1));
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[(rr + j) * GPITCH + kk] = uint16_t(v[j >> 1] >> (16 * (j & 1)));
  }
}

template <bool BF16>
__global__ __launch_bounds__(GT) void k_gemm16(Operand A, Operand B, uint16_t *__restrict__ C, int M, int N, int K,
                                              int ldc, float alpha, float beta) {
  __shared__ __align__(16) uint16_t As[2][GBM * GPITCH], Bs[2][GBN * GPITCH];
  const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const int chunks = (K + GBK - 1) / GBK;
  stage(A, m0, 0, K, As[0]);
  stage(B, n0, 0, K, Bs[0]);
  __syncthreads();
  for (int c = 0; c < chunks; ++c) {
    const int cur = c & 1;
    if (c + 1 < chunks) {   // the next chunk goes to the other buffer while this one is multiplied
      stage(A, m0, (c + 1) * GBK, K, As[cur ^ 1]);
      stage(B, n0, (c + 1) * GBK, K, Bs[cur ^ 1]);
    }
    const uint16_t *a = As[cur] + (wm + (lane & 31)) * GPITCH + 8 * (lane >> 5);
    const uint16_t *b = Bs[cur] + (wn + (lane & 31)) * GPITCH + 8 * (lane >> 5);
#pragma unroll
    for (int ks = 0; ks < GBK / 16; ++ks)
      acc = mfma16<BF16>(*reinterpret_cast<const u32x4 *>(a + 16 * ks), *reinterpret_cast<const u32x4 *>(b + 16 * ks), acc);
    __syncthreads();
  }
  // accumulator v of lane l: row 8 * (v / 4) + 4 * (l / 32) + v % 4, column l % 32 of the wavefront's quarter
  const int col = n0 + wn + (lane & 31);
  if (col < N) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = m0 + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (row < M) {
        uint16_t *dst = C + size_t(row) * ldc + col;
        float r = alpha * acc[v];
        if (beta != 0.f) r += beta * (BF16 ? sgh_bf16_to_f32(*dst) : sgh_f16_to_f32(*dst));
        *dst = BF16 ? sgh_f32_to_bf16(r) : sgh_f32_to_f16(r);
      }
    }
  }
}

// ---- few output tiles: the reduction split over the wavefronts of a workgroup ----------------------------------------
// As in gemm_split.hip: a workgroup owns a T x T tile of C (T = 32: v_mfma_f32_32x32x16, T = 16: v_mfma_f32_16x16x32), its W
// wavefronts a W-th of the reduction each, fed from global memory without LDS, and the partial tiles are added in wavefront
// order.  Lane (i, h) supplies reduction indices 8 h .. 8 h + 7 of a group for row / column i of its operand.  With the
// reduction index contiguous that is one 16-byte load.  With the row index contiguous it would be eight 2-byte loads of a
// column, each as dear as a 16-byte one; instead the even lane of a pair loads the dwords (two columns) of rows 0..3 and the
// odd lane those of rows 4..7, each packs its own and its neighbour's column with v_perm_b32, and the halves change lanes.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

template <bool KC>
struct Feed16 {
  rsrc_t r;
  int off;    // byte offset of the lane's first load at reduction index 8 h; refused by the buffer when the row does not exist
  int col;    // byte offset of the lane's own row at reduction index 8 h, or refused
  int ld;     // bytes
  bool odd, single;   // single: this tile holds the last row of an odd number of rows, where the pair loads would read past it
  __device__ __forceinline__ Feed16(const uint16_t *p, int ld_, unsigned bytes, int row0, int i, int rows, int h, int tile) {
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p), 0, bytes, 0x00020000);
    ld = ld_ * 2;
    odd = i & 1;
    const int row = row0 + i;
    col = row < rows ? (KC ? row * ld + 16 * h : 8 * h * ld + row * 2) : int(0x80000000u);
    single = !KC && (rows & 1) && row0 + tile >= rows;
    off = KC ? col : (row & ~1) < rows ? (8 * h + (odd ? 4 : 0)) * ld + (row & ~1) * 2 : int(0x80000000u);
  }
  struct Raw {
    u32x4 v;
  };
  __device__ __forceinline__ Raw request(int k) const {   // (k uniform, the whole group inside)
    Raw w;
    if constexpr (KC) w.v = __builtin_amdgcn_raw_buffer_load_b128(r, off, k * 2, 0);
    else
#pragma unroll
      for (int u = 0; u < 4; ++u) w.v[u] = __builtin_amdgcn_raw_buffer_load_b32(r, off, (k + u) * ld, 0);
    return w;
  }
  __device__ __forceinline__ u32x4 octet(const Raw &w) const {
    if constexpr (KC) return w.v;
    // halves of two dwords: 0x05040100 the low ones, 0x07060302 the high ones
    const unsigned own = odd ? 0x07060302u : 0x05040100u, other = odd ? 0x05040100u : 0x07060302u;
    const u32x2 mine = {__builtin_amdgcn_perm(w.v[1], w.v[0], own), __builtin_amdgcn_perm(w.v[3], w.v[2], own)};
    u32x2 theirs = {__builtin_amdgcn_perm(w.v[1], w.v[0], other), __builtin_amdgcn_perm(w.v[3], w.v[2], other)};
#pragma unroll
    for (int e = 0; e < 2; ++e)   // (quad_perm 1, 0, 3, 2: the neighbour's)
      theirs[e] = __builtin_amdgcn_update_dpp(0u, theirs[e], 0xB1, 0xF, 0xF, false);
    return odd ? u32x4{theirs[0], theirs[1], mine[0], mine[1]} : u32x4{mine[0], mine[1], theirs[0], theirs[1]};
  }
  // element by element: the group that K ends in (`left` of this lane's eight indices exist) and tiles marked `single`
  __device__ __forceinline__ u32x4 elements(int k, int left) const {
    u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int o = u < left && col >= 0 ? col + (KC ? (k + u) * 2 : (k + u) * ld) : int(0x80000000u);
      v[u >> 1] |= unsigned(__builtin_amdgcn_raw_buffer_load_b16(r, o, 0, 0)) << (16 * (u & 1));
    }
    return v;
  }
};

template <bool BF16, int T>
struct Mfma16;
template <bool BF16>
struct Mfma16<BF16, 32> {
  typedef f32x16 acc;
  static __device__ __forceinline__ acc run(u32x4 a, u32x4 b, acc c) { return mfma16<BF16>(a, b, c); }
  static __device__ __forceinline__ int row(int v, int h) { return 8 * (v >> 2) + 4 * h + (v & 3); }   // of accumulator v
};
template <bool BF16>
struct Mfma16<BF16, 16> {
  typedef f32x4 acc;
  static __device__ __forceinline__ acc run(u32x4 a, u32x4 b, acc c) {
    if constexpr (BF16)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int v, int h) { return 4 * h + v; }
};

template <bool BF16, bool AK, bool BKc, int T, int W>
__global__ __launch_bounds__(W * 64) void k_gemm16_split(const uint16_t *__restrict__ A, int lda, unsigned a_bytes,
                                                         const uint16_t *__restrict__ B, int ldb, unsigned b_bytes,
                                                         uint16_t *__restrict__ C, int ldc, int M, int N, int K, int kq,
                                                         float alpha, float beta) {
  __shared__ float part[W][T * T];
  typedef Mfma16<BF16, T> MM;
  constexpr int G = 8 * (64 / T);   // reduction indices of a group: eight per lane
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, i = lane % T, h = lane / T;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int kb = __builtin_amdgcn_readfirstlane(wave * kq), ke = kb + kq < K ? kb + kq : K;   // (kq is a multiple of G)
  const Feed16<AK> fa(A, lda, a_bytes, m0, i, M, h, T);
  const Feed16<BKc> fb(B, ldb, b_bytes, n0, i, N, h, T);
  typename MM::acc acc;
#pragma unroll
  for (int v = 0; v < T * T / 64; ++v) acc[v] = 0.f;
  int k = kb;
  if (!fa.single && !fb.single) {
    constexpr int U = 4;   // groups requested before the first is used
    for (; k + G * U <= ke; k += G * U) {
      typename Feed16<AK>::Raw a[U];
      typename Feed16<BKc>::Raw b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = fa.request(k + G * u), b[u] = fb.request(k + G * u);
#pragma unroll
      for (int u = 0; u < U; ++u) acc = MM::run(fa.octet(a[u]), fb.octet(b[u]), acc);
    }
    for (; k + G <= ke; k += G) {
      const typename Feed16<AK>::Raw a = fa.request(k);
      const typename Feed16<BKc>::Raw b = fb.request(k);
      acc = MM::run(fa.octet(a), fb.octet(b), acc);
    }
  }
  for (; k < ke; k += G) acc = MM::run(fa.elements(k, ke - k - 8 * h), fb.elements(k, ke - k - 8 * h), acc);
#pragma unroll
  for (int v = 0; v < T * T / 64; ++v) part[wave][MM::row(v, h) * T + i] = acc[v];
  __syncthreads();
#pragma unroll
  for (int e = t; e < T * T; e += W * 64) {
    float v = part[0][e];
#pragma unroll
    for (int w = 1; w < W; ++w) v += part[w][e];
    const int row = e / T, col = e % T;
    if (m0 + row < M && n0 + col < N) {
      uint16_t *dst = C + size_t(m0 + row) * ldc + n0 + col;
      float r = alpha * v;
      if (beta != 0.f) r += beta * (BF16 ? sgh_bf16_to_f32(*dst) : sgh_f16_to_f32(*dst));
      *dst = BF16 ? sgh_f32_to_bf16(r) : sgh_f32_to_f16(r);
    }
  }
}

template <bool BF16, bool AK, bool BKc>
void launch_split(int tile, int waves, const uint16_t *A, int lda, const uint16_t *B, int ldb, uint16_t *C, int ldc, int M, int N,
                  int K, float alpha, float beta, hipStream_t s) {
  const int G = 512 / tile, kq = ((K + waves - 1) / waves + G - 1) / G * G;
  const unsigned ab = unsigned((size_t(AK ? M - 1 : K - 1) * lda + (AK ? K : M)) * 2);
  const unsigned bb = unsigned((size_t(BKc ? N - 1 : K - 1) * ldb + (BKc ? K : N)) * 2);
  const dim3 grid((N + tile - 1) / tile, (M + tile - 1) / tile);
#define SGH_SPLIT_CASE(T_, W_)                                                                                                      \
  hipLaunchKernelGGL((k_gemm16_split<BF16, AK, BKc, T_, W_>), grid, dim3(W_ * 64), 0, s, A, lda, ab, B, ldb, bb, C, ldc, M, N, K,   \
                     kq, alpha, beta)
  if (tile == 16 && waves == 8) SGH_SPLIT_CASE(16, 8);
  else if (tile == 16) SGH_SPLIT_CASE(16, 4);
  else if (waves == 8) SGH_SPLIT_CASE(32, 8);
  else SGH_SPLIT_CASE(32, 4);
#undef SGH_SPLIT_CASE
}

// Whether the split kernel takes the problem, its tile and the wavefronts that share one.  Measured in binary16 (us, tiled
// kernel / 32-wide / 16-wide tiles, 8 wavefronts; NN = neither operand transposed, NT = B transposed):
//   256 x 1000 x 2048 NN    42 / 10.2 / 19        128 x 10 x 4096 NN    133 / 13.5 / 8.9
//   1024 x 1024 x 1024 NN   23 / 17.3, NT 16.9 / 16.9    four 32-wide tiles per CU;
//   1000 x 2048 x 512 NN    14.5 / 17.2                  eight: the tiled kernel loads half the bytes per product
// 16-wide tiles win while 32-wide ones leave half of the CUs without a workgroup; four wavefronts are enough for short
// reductions (784 x 1000 x 128: 5.0 / 5.1 us with 4 / 8), 16 gain nothing over 8 (512 x 1024 x 2048: 17.6 / 17.5).
bool split_plan(int M, int N, int K, int *tile, int *waves) {
  const long t32 = long((M + 31) / 32) * ((N + 31) / 32), cus = sgh_num_cus();
  if (t32 > 4 * cus) return false;
  *tile = 2 * t32 < cus ? 16 : 32;
  *waves = K < 256 ? 4 : 8;
  return (M + *tile - 1) / *tile <= 65535;
}

template <bool BF16>
int gemm16(int transA, int transB, int M, int N, int K, float alpha, const uint16_t *A, int lda, const uint16_t *B, int ldb,
           float beta, uint16_t *C, int ldc, void *stream) {
  if (M < 0 || N < 0 || K < 0) return SGH_EINVAL;
  if (M == 0 || N == 0) return SGH_OK;
  if (!C || ldc < N || (K > 0 && (!A || !B))) return SGH_EINVAL;
  // pitches of the stored matrices: A is [M][K] (transposed: [K][M]), B is [K][N] (transposed: [N][K])
  if (K > 0 && (lda < (transA ? M : K) || ldb < (transB ? K : N))) return SGH_EINVAL;
  const Operand a{A, lda, transA ? 0 : 1, sgh_aligned16(A) && lda % 8 == 0, M};
  const Operand b{B, ldb, transB ? 1 : 0, sgh_aligned16(B) && ldb % 8 == 0, N};
  const dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM);
  if (grid.y > 65535u) return SGH_EUNSUPPORTED;
  hipStream_t st = sgh_stream_of(stream);
  sgh_prof_scope prof("gemm16", 2.0 * M * N * K, st);
  int tile, waves;
  if (K > 0 && split_plan(M, N, K, &tile, &waves) && size_t(transA ? K : M) * lda < (size_t(1) << 30) &&
      size_t(transB ? N : K) * ldb < (size_t(1) << 30)) {   // (operands addressed with 32-bit byte offsets)
    if (!transA && transB) launch_split<BF16, true, true>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else if (!transA) launch_split<BF16, true, false>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else if (transB) launch_split<BF16, false, true>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else launch_split<BF16, false, false>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    SGH_LAUNCH_CHECK();
    return SGH_OK;
  }
  hipLaunchKernelGGL(k_gemm16<BF16>, grid, dim3(GT), 0, st, a, b, C, M, N, K, ldc, alpha, beta);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}

}  // namespace

extern "C" {

int sgh_gemm_f16(int transA, int transB, int M, int N, int K, float alpha, const uint16_t *A, int lda, const uint16_t *B,
                 int ldb, float beta, uint16_t *C, int ldc, void *stream) {
  return gemm16<false>(transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, stream);
}
int sgh_gemm_bf16(int transA, int transB, int M, int N, int K, float alpha, const uint16_t *A, int lda, const uint16_t *B,
                  int ldb, float beta, uint16_t *C, int ldc, void *stream) {
  return gemm16<true>(transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, stream);
}

}  // extern "C"
