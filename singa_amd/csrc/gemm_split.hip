// fp32 GEMM for few output tiles: C = alpha * op(A) * op(B) + beta * C with the reduction split over the wavefronts of a
// workgroup (the dense layers: a batch of rows against a few to a few thousand columns).
//
// Such a problem is bound by latency, not by bandwidth or the matrix pipe: 128 x 4096 x 10 is 10 MFLOP on 2 MB.  The tiled
// kernel walked the whole reduction in two workgroups, 16 indices per barrier (135 us).  Here a workgroup owns a 32 x 32
// (or 16 x 16) tile of C and its W wavefronts each take a W-th of the reduction, feeding v_mfma_f32_32x32x2_f32 straight from global
// memory: lane (i, h) supplies A[i][h] and B[h][i], so it takes reduction indices 8 j + 4 h + (0..3) of row / column i of
// each operand -- one 16-byte load where the reduction index is the contiguous one, four dwords (32 lanes: 128 contiguous
// bytes) where it is not -- and the four instructions of group j consume the pairs (8 j + u, 8 j + 4 + u).  The W partial
// tiles are added in wavefront order through LDS, so results are the same on every run.
// What it measures stands beside `plan`.
#include "common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

// One operand: element (row, k) at p[row * ld + k] (KC: reduction index contiguous) or p[k * ld + row].
template <bool KC>
struct Feed {
  rsrc_t r;
  int off;   // byte offset of the lane's row at reduction index 4 h (h: lane / T); refused by the buffer when the row does not exist
  int ld;    // bytes
  __device__ __forceinline__ Feed(const float *p, int ld_, unsigned bytes, int row, bool ok, int h) {
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, bytes, 0x00020000);
    ld = ld_ * 4;
    off = ok ? (KC ? row * ld + 16 * h : 4 * h * ld + row * 4) : int(0x80000000u);
  }
  __device__ __forceinline__ f32x4 load(int k) const {   // (k uniform, the whole group inside)
    if constexpr (KC) return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, k * 4, 0));
    f32x4 v;
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, (k + u) * ld, 0));
    return v;
  }
  // the group that K ends in: `left` of this lane's four indices exist
  __device__ __forceinline__ f32x4 load_tail(int k, int left) const {
    f32x4 v;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int o = u < left && off >= 0 ? off + (KC ? (k + u) * 4 : (k + u) * ld) : int(0x80000000u);
      v[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
    }
    return v;
  }
};

template <int T>
struct Mfma;
template <>
struct Mfma<32> {
  typedef f32x16 acc;
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int v, int h) { return 8 * (v >> 2) + 4 * h + (v & 3); }   // of accumulator v
};
template <>
struct Mfma<16> {
  typedef f32x4 acc;
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int v, int h) { return 4 * h + v; }
};

// out[n] = sum over the rows of m[row][n], in ascending order, of the T columns from n0 on: 32 loads in flight per column
template <int T>
__device__ __forceinline__ void sum_columns(const float *__restrict__ m, int ld, int rows, int cols, int n0, float *__restrict__ out) {
  const int j = n0 + int(threadIdx.x);
  if (threadIdx.x >= T || j >= cols) return;
  constexpr int U = 32;
  float s = 0.f;
  int i = 0;
  for (; i + U <= rows; i += U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = m[size_t(i + u) * ld + j];
#pragma unroll
    for (int u = 0; u < U; ++u) s += v[u];
  }
  for (; i < rows; ++i) s += m[size_t(i) * ld + j];
  out[j] = s;
}

// (AROUND: `around` is not empty.  Its tests in the plain product's store cost every fp32 GEMM 0.2 to 0.5 us)
template <bool AK, bool BKc, int T, int W, bool AROUND>
__global__ __launch_bounds__(W * 64) void k_gemm_split(const float *__restrict__ A, int lda, unsigned a_bytes,
                                                       const float *__restrict__ B, int ldb, unsigned b_bytes,
                                                       float *__restrict__ C, long ldc, int M, int N, int K, int kq, float alpha,
                                                       float beta, sgh_gemm_around around) {
  if constexpr (AROUND && !BKc) {
    if (around.colsum && blockIdx.y == gridDim.y - 1) {   // (a row of workgroups of its own, beside the tiles)
      sum_columns<T>(B, ldb, K, N, blockIdx.x * T, around.colsum);
      return;
    }
  }
  __shared__ float part[W][T * T];
  constexpr int G = 4 * (64 / T);   // reduction indices of a group: four per lane
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, i = lane % T, h = lane / T;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int kb = __builtin_amdgcn_readfirstlane(wave * kq), ke = kb + kq < K ? kb + kq : K;   // (kq is a multiple of G)
  const Feed<AK> fa(A, lda, a_bytes, m0 + i, m0 + i < M, h);
  const Feed<BKc> fb(B, ldb, b_bytes, n0 + i, n0 + i < N, h);
  typename Mfma<T>::acc acc;
#pragma unroll
  for (int v = 0; v < T * T / 64; ++v) acc[v] = 0.f;
  constexpr int U = 4;   // groups requested before the first is used
  int k = kb;
  for (; k + G * U <= ke; k += G * U) {
    f32x4 a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = fa.load(k + G * u), b[u] = fb.load(k + G * u);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = Mfma<T>::run(a[u][e], b[u][e], acc);
  }
  for (; k + G <= ke; k += G) {
    const f32x4 a = fa.load(k), b = fb.load(k);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = Mfma<T>::run(a[e], b[e], acc);
  }
  if (k < ke) {
    const f32x4 a = fa.load_tail(k, ke - k - 4 * h), b = fb.load_tail(k, ke - k - 4 * h);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = Mfma<T>::run(a[e], b[e], acc);
  }
#pragma unroll
  for (int v = 0; v < T * T / 64; ++v) part[wave][Mfma<T>::row(v, h) * T + i] = acc[v];
  __syncthreads();
#pragma unroll
  for (int e = t; e < T * T; e += W * 64) {
    float v = part[0][e];
#pragma unroll
    for (int w = 1; w < W; ++w) v += part[w][e];
    const int row = e / T, col = e % T;
    if (m0 + row < M && n0 + col < N) {
      float *p = C + size_t(m0 + row) * ldc + n0 + col;
      float r = beta == 0.f ? alpha * v : alpha * v + beta * *p;
      if constexpr (AROUND) {
        if (around.bias) r += around.bias[n0 + col];
        if (around.relu) r = r >= 0.f ? r : 0.f;
        if (around.gate) r = around.gate[size_t(m0 + row) * N + n0 + col] > 0.f ? r : 0.f;
      }
      *p = r;
    }
  }
}

template <bool AK, bool BKc>
void launch(int tile, int waves, const float *A, int lda, const float *B, int ldb, float *C, int ldc, int M, int N, int K, float alpha,
            float beta, const sgh_gemm_around &around, hipStream_t s) {
  const int G = 256 / tile, kq = ((K + waves - 1) / waves + G - 1) / G * G;
  const unsigned ab = unsigned((size_t(AK ? M - 1 : K - 1) * lda + (AK ? K : M)) * 4);
  const unsigned bb = unsigned((size_t(BKc ? N - 1 : K - 1) * ldb + (BKc ? K : N)) * 4);
  const dim3 grid((N + tile - 1) / tile, (M + tile - 1) / tile + (around.colsum ? 1 : 0));
  const bool plain = !around.bias && !around.gate && !around.colsum && !around.relu;
#define SGH_SPLIT_KERNEL(T_, W_, AROUND_)                                                                                           \
  hipLaunchKernelGGL((k_gemm_split<AK, BKc, T_, W_, AROUND_>), grid, dim3(W_ * 64), 0, s, A, lda, ab, B, ldb, bb, C, long(ldc), M,  \
                     N, K, kq, alpha, beta, around)
#define SGH_SPLIT_CASE(T_, W_)                                \
  do {                                                        \
    if (plain) SGH_SPLIT_KERNEL(T_, W_, false);               \
    else if constexpr (AK || !BKc) SGH_SPLIT_KERNEL(T_, W_, true);   /* (no layer has both operands transposed) */ \
  } while (0)
  if (tile == 16 && waves == 8) SGH_SPLIT_CASE(16, 8);
  else if (tile == 16) SGH_SPLIT_CASE(16, 4);
  else if (waves == 16) SGH_SPLIT_CASE(32, 16);
  else if (waves == 8) SGH_SPLIT_CASE(32, 8);
  else SGH_SPLIT_CASE(32, 4);
#undef SGH_SPLIT_KERNEL
#undef SGH_SPLIT_CASE
}

}  // namespace

// Whether the split kernel takes the problem, its tile and the wavefronts that share one.  Measured (us, tiled kernel before /
// 32-wide tiles / 16-wide tiles; NN = neither operand transposed, NT = B transposed):
//   128 x 10 x 4096 NN      135 / 25 / 16       16-wide tiles win while 32-wide ones leave half of the CUs without a
//   128 x 1000 x 784 NN      30 / 7.5 / 7.2     workgroup (they load twice the bytes per product: 256 x 1000 x 2048 NN
//   256 x 1000 x 2048 NN     71 / 14 / 28       is the far side of that line)
//   1000 x 2048 x 512 NN     29 / 24 / 38       eight 32-wide tiles per CU, 2048 x 4096 x 512 NN 91 / 88: beyond eight
//   2048 x 1000 x 128 NN    11.8 / 10.2         the tiled kernel's reuse of its operands in LDS takes over
//   512 x 1024 x 2048 NT     60 / 33            with both reductions contiguous a wavefront's 16-byte loads touch 32 rows,
//   1000 x 2048 x 512 NT     27 / 31            so the line lies at three tiles per CU
// Wavefronts: 16 pay from a reduction of 1024 on (512 x 1024 x 2048 NN: 28 / 25 / 24 us with 4 / 8 / 16), and with few
// indices per wavefront the sum of the partial tiles costs more than it saves (784 x 1000 x 128 NN: 6.1 / 6.0 / 7.1).
// Reductions of 1 to 128 take it as well: 4.2 us on either kernel at 128 x 1000 x 16, 4.7 / 4.8 at 1024 x 1024 x 16, 4.7 / 4.2
// at 2048 x 512 x 4 and 5.6 / 4.4 at 512 x 512 x 64.
//   Beyond five and a half tiles per CU long reductions go back to the tiled kernel: NN 421 x 3758 x 1172 63 / 74, 1809 x 947 x
// 1833 96 / 109, TT 848 x 2072 x 2733 137 / 175 against 30 / 22 at 1879 x 625 x 529 and 33 / 33 at 773 x 1988 x 585; with A alone
// transposed it holds on to reductions of 2000 (1672 x 925 x 2032 104 / 79; 503 x 3847 x 2373 124 / 131).
//   With both reductions contiguous four wavefronts do from one tile per CU on, eight before: 160 problems, reductions of 256 to
// 4096, against the kernels before; from one tile per CU on 0.91 to 1.08 times as fast with the wavefronts of the other cases and
// 1.01 to 1.11 with four (392 x 677 x 3084: 41.8 us before, 55.6, 42); below, 2048 and up, 1.20 with sixteen and 1.22 with eight.
static bool plan(bool ta, bool tb, int M, int N, int K, int *tile, int *waves) {
  const bool nt = !ta && tb;
  const long t32 = long((M + 31) / 32) * ((N + 31) / 32), cus = sgh_num_cus();
  if (t32 > (nt ? 3 : 8) * cus || (2 * t32 > 11 * cus && K > (ta && !tb ? 2048 : 640))) return false;
  *tile = 2 * t32 < cus ? 16 : 32;
  *waves = K < 256 ? 4 : K < 1024 || *tile == 16 ? 8 : 16;
  if (nt && *tile == 32 && K >= 256) *waves = t32 >= cus ? 4 : 8;
  return (M + *tile - 1) / *tile < 65535;   // (one more row of workgroups sums columns)
}

int sgh_gemm_split_run(int transA, int transB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb,
                       float beta, float *C, int ldc, const sgh_gemm_around &around, hipStream_t s) {
  int tile, waves;
  if (!plan(transA, transB, M, N, K, &tile, &waves)) return SGH_EUNSUPPORTED;
  if (!transA && transB) launch<true, true>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, around, s);
  else if (!transA) launch<true, false>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, around, s);
  else if (transB) launch<false, true>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, around, s);
  else launch<false, false>(tile, waves, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, around, s);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}
