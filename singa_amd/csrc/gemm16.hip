// GEMM on 16-bit matrices (binary16 / bfloat16): C = alpha * op(A) * op(B) + beta * C with fp32
// accumulation on v_mfma_f32_32x32x16_{f16,bf16} and one rounding at the store -- the Linear layers of
// a half model (the reference calls cublasHgemm: src/core/tensor/tensor_math_cuda.h:1163-1187).
//
// Three kernels; none splits the reduction over workgroups and every sum is taken in a fixed order: results are run-to-run
// identical.  k_gemm16_tile (many output tiles) and k_gemm16_split (few) do the work; k_gemm16 is left with what neither can
// address: operands of 2 GB and more, 2^24 tiles, and fewer than eight rows, columns or reduction indices against many of the others.
//
// k_gemm16: a workgroup of four wavefronts owns a 64 x 64 tile of C, a wavefront a 32 x 32 quarter.  Both matrix
// operands want, per lane, eight consecutive reduction indices of one tile row, so both LDS tiles are
// [row][k] with k contiguous (pitch 32 + 8 halves: 16-byte reads without bank conflicts).  With k contiguous in memory
// a thread copies one octet with a 16-byte load; with the row index contiguous
// it loads eight rows of one k with a 16-byte load and writes them as eight 2-byte LDS
// stores; pointers, pitches or edges that do not allow the 16-byte access fall back to single elements.
#include <hip/hip_runtime.h>

#include <type_traits>

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

// ---- many output tiles -----------------------------------------------------------------------------------------------
// A workgroup of four wavefronts owns a BT x BT tile of C (BT = 64 or 128, a wavefront a quarter).  Chunks of 64 reduction
// indices go through two register sets (requested two chunks ahead) into two LDS buffers, one barrier per chunk.
// A tile is kept in LDS as it lies in memory: [row][k] where the reduction index is the contiguous one (16-byte reads are the
// fragments), [k][row] where the row is (ds_read_b64_tr_b16 hands a lane four k of its row).  Either way a load is 16 bytes of
// one line of the matrix at any element alignment.  Rows come in octets, the last of which ends with the matrix and overlaps its
// neighbour (nothing is read beyond an operand, no masks); reduction indices beyond K are zeros: whole lines where k is a line,
// else the last octet ends with K too and is shifted down.
//   Bound by the serial phases of a chunk (request, 16 KB to LDS, 32 KB from it, 64 matrix instructions: 0.33 us with a CU to
// itself), not by the loads: four register sets instead of two were 5-10 % slower.  So several workgroups per CU, or two groups of
// four wavefronts that take alternate chunks and add their sums in order.  bfloat16, before (k_gemm16 or k_gemm16_split) -> now, us:
// 256 x 2048 x 1000 NT 9.8 -> 6.7, 2048 x 1000 x 256 TN 12.1 -> 5.6, 1024^3 NN 16.8 -> 7.0, 1001 x 2049 x 333 NN 31.8 -> 9.4, 1500^3 NT
// 169 -> 23, 2048 x 4096 x 1200 NT 71 -> 30 (670 TFLOP/s).  An empty launch is 3.7 of each.
constexpr int TK = 64, NOT_THERE = int(0x80000000u);

template <bool KC, int BT>
struct Panel {
  static constexpr int N = BT / 32;   // 16-byte loads of a thread and chunk
  rsrc_t r;
  int off[KC ? N : 1];   // byte offset of the thread's loads at reduction index 0 (rows apart) / of its first line
  int ld2, K, k;         // pitch in bytes; the thread's own reduction index in a chunk
  u32x4 v[2][N];
  __device__ __forceinline__ void init(const uint16_t *p, int ld, unsigned bytes, int row0, int rows, int K_) {
    const int t = threadIdx.x & 255;
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p), 0, bytes, 0x00020000);
    ld2 = ld * 2, K = K_;
    if constexpr (KC) {
      k = (t & 7) * 8;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int row = row0 + 32 * j + (t >> 3), base = min(row & ~7, rows - 8);
        off[j] = (base + (row & 7)) * ld2 + k * 2;
      }
    } else {
      k = t / (BT / 8);
      off[0] = k * ld2 + min(row0 + (t % (BT / 8)) * 8, rows - 8) * 2;
    }
  }
  template <int S>
  __device__ __forceinline__ void request(int k0) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if constexpr (KC) {
        const int over = k0 + k + 8 - K;   // beyond K: the octet that ends with K, or nothing
        v[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, over >= 8 ? NOT_THERE : off[j] + 2 * (k0 - max(over, 0)), 0, 0));
      } else {
        constexpr int LINES = 256 / (BT / 8);
        v[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, k0 + k + LINES * j < K ? off[0] + LINES * j * ld2 : NOT_THERE, k0 * ld2, 0));
      }
    }
  }
  template <int S>
  __device__ __forceinline__ void stage(uint16_t *tile, int k0) {
    const int t = threadIdx.x & 255;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if constexpr (KC) {
        const int row = 32 * j + (t >> 3);
        u32x4 w = v[S][j];
        if (k0 + TK > K) {   // (uniform: the last chunk)
          const int over = k0 + k + 8 - K;
          if (over > 0 && over < 8) {
            if (over & 4) w = u32x4{w[2], w[3], 0u, 0u};
            if (over & 2) w = u32x4{w[1], w[2], w[3], 0u};
            if (over & 1)
              w = u32x4{__builtin_amdgcn_alignbyte(w[1], w[0], 2), __builtin_amdgcn_alignbyte(w[2], w[1], 2),
                        __builtin_amdgcn_alignbyte(w[3], w[2], 2), w[3] >> 16};
          }
        }
        *reinterpret_cast<u32x4 *>(tile + row * TK + (((t & 7) ^ ((row >> 1) & 7)) * 8)) = w;
      } else {
        const int line = k + 256 / (BT / 8) * j, oct = t % (BT / 8);
        *reinterpret_cast<u32x4 *>(tile + line * BT + (oct ^ (BT == 64 ? (line & 2) << 1 : (line & 3) << 2)) * 8) = v[S][j];
      }
    }
  }
  // fragments of 32-row tile `tile32` for matrix steps k2 and k2 + 1 (16 reduction indices each)
  static __device__ __forceinline__ void fragments(const uint16_t *tile, int tile32, int k2, u32x4 (&f)[2]) {
    const int lane = threadIdx.x & 63, lh = lane >> 5;
    if constexpr (KC) {
      const int row = 32 * tile32 + (lane & 31);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        f[s] = *reinterpret_cast<const u32x4 *>(tile + row * TK + (((2 * (k2 + s) + lh) ^ ((row >> 1) & 7)) * 8));
    } else {
      typedef __attribute__((address_space(3))) const uint16_t lds_u16;
      const int line = (lane >> 2) & 3, oct = 4 * tile32 + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
      const unsigned a = unsigned(size_t((lds_u16 *)(tile + (16 * k2 + 8 * lh + line) * BT +
                                                     (oct ^ (BT == 64 ? (line & 2) << 1 : line << 2)) * 8 + (lane & 1) * 4)));
      u32x2 q[4];
      // (one block with its own wait: the builtin waits for every load under way)
      if constexpr (BT == 64)
        asm volatile(
            "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %4 offset:512\n\t"
            "ds_read_b64_tr_b16 %2, %4 offset:2048\n\tds_read_b64_tr_b16 %3, %4 offset:2560\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]) : "v"(a) : "memory");
      else
        asm volatile(
            "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %4 offset:1024\n\t"
            "ds_read_b64_tr_b16 %2, %4 offset:4096\n\tds_read_b64_tr_b16 %3, %4 offset:5120\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]) : "v"(a) : "memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) f[s] = u32x4{q[2 * s][0], q[2 * s][1], q[2 * s + 1][0], q[2 * s + 1][1]};
    }
  }
};

template <bool BF16, bool AK, bool BKc, int BT, int KS>
__global__ __launch_bounds__(256 * KS) void k_gemm16_tile(const uint16_t *__restrict__ A, int lda, unsigned a_bytes,
                                                     const uint16_t *__restrict__ B, int ldb, unsigned b_bytes,
                                                     uint16_t *__restrict__ C, int ldc, int M, int N, int K, int mtiles, int tiles,
                                                     float alpha, float beta) {
  constexpr int TM = BT / 64, HALF = BT * TK, OP = BT + 8;
  static_assert(OP * BT <= 4 * HALF && 2 * BT * BT <= 4 * HALF, "");
  __shared__ __align__(16) uint16_t lds_all[KS][2][2 * HALF];
  // workgroup w runs on XCD w % 8: an XCD takes neighbouring tiles, which share their panels in its L2
  const int per = (tiles + 7) >> 3, l = (int(blockIdx.x) & 7) * per + (int(blockIdx.x) >> 3);
  if ((int(blockIdx.x) >> 3) >= per || l >= tiles) return;
  const int m0 = (l % mtiles) * BT, n0 = (l / mtiles) * BT;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = (wave >> 1) & 1, wn = wave & 1;
  const int group = wave >> 2;   // of four wavefronts: chunks group, group + KS, ...
  uint16_t (*const lds)[2 * HALF] = lds_all[group];
  Panel<AK, BT> pa;
  Panel<BKc, BT> pb;
  pa.init(A, lda, a_bytes, m0, M, K);
  pb.init(B, ldb, b_bytes, n0, N, K);
  f32x16 acc[TM][TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  auto multiply = [&](const uint16_t *st) {
#pragma unroll
    for (int k2 = 0; k2 < TK / 16; k2 += 2) {
      u32x4 fa[TM][2], fb[TM][2];
#pragma unroll
      for (int i = 0; i < TM; ++i) Panel<AK, BT>::fragments(st, wm * TM + i, k2, fa[i]);
#pragma unroll
      for (int i = 0; i < TM; ++i) Panel<BKc, BT>::fragments(st + HALF, wn * TM + i, k2, fb[i]);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) acc[i][j] = mfma16<BF16>(fb[j][s], fa[i][s], acc[i][j]);   // rows: n, columns: m
    }
  };
  const int rounds = (K + KS * TK - 1) / (KS * TK), kg = group * TK;
  auto at = [&](int c) { return c * (KS * TK) + kg; };   // first reduction index of the group's chunk c (beyond K: zeros)
  auto request = [&](auto SET, int c) {
    constexpr int S = decltype(SET)::value;
    pa.template request<S>(at(c)), pb.template request<S>(at(c));
  };
  auto stage = [&](auto SET, int c) {
    constexpr int S = decltype(SET)::value;
    pa.template stage<S>(lds[S], at(c)), pb.template stage<S>(lds[S] + HALF, at(c));
  };
  // chunk c of the group: request what takes its registers, multiply, hand the next one to the other buffer; false at the end
  auto step = [&](auto SET, int c) {
    constexpr int S = decltype(SET)::value;
    __syncthreads();
    request(SET, c + 2);
    multiply(lds[S]);
    if (c + 1 >= rounds) return false;
    stage(std::integral_constant<int, S ^ 1>{}, c + 1);
    return true;
  };
  typedef std::integral_constant<int, 0> Set0;
  typedef std::integral_constant<int, 1> Set1;
  request(Set0{}, 0);
  request(Set1{}, 1);
  stage(Set0{}, 0);
  for (int c = 0; step(Set0{}, c) && step(Set1{}, c + 1); c += 2) {
  }
  if constexpr (KS > 1) {   // the groups' sums in their order
    static_assert(BT == 64, "");
    __syncthreads();
    float *const part = reinterpret_cast<float *>(lds_all[group]) + (wave & 3) * 1024;
#pragma unroll
    for (int v = 0; v < 16; ++v) part[v * 64 + lane] = acc[0][0][v];
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int g = 1; g < KS; ++g)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[0][0][v] += reinterpret_cast<const float *>(lds_all[g])[(wave & 3) * 1024 + v * 64 + lane];
    }
  }
  // the tile leaves through LDS as [m][n] rows of octets; a lane holds four neighbouring n of one m
  __syncthreads();
  uint16_t *const o = lds_all[0][0];
  if (group == 0)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int v = 0; v < 16; v += 4) {
        const int row = (wm * TM + i) * 32 + (lane & 31), col = (wn * TM + j) * 32 + 2 * v + 4 * (lane >> 5);
        const int gm = min((m0 + row) & ~7, M - 8) + (row & 7), gn = min((n0 + col) & ~7, N - 8) + (col & 7);
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = alpha * acc[i][j][v + e];
        }
        if (beta != 0.f) {   // (an element of two octets is stored by the first of them only, below)
          const uint16_t *c = C + size_t(gm) * ldc + gn;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += beta * (BF16 ? sgh_bf16_to_f32(c[e]) : sgh_f16_to_f32(c[e]));
        }
        const u32x2 q = BF16 ? u32x2{sgh_pack2_bf16(x[0], x[1]), sgh_pack2_bf16(x[2], x[3])}
                             : u32x2{sgh_pack2_f16(x[0], x[1]), sgh_pack2_f16(x[2], x[3])};
        *reinterpret_cast<u32x2 *>(o + row * OP + col) = q;
      }
  __syncthreads();
  constexpr int OCT = BT / 8, STEP = 256 * KS / OCT;
#pragma unroll
  for (int row = t / OCT; row < BT; row += STEP) {
    const int go = n0 + (t % OCT) * 8;
    const int gm = min((m0 + row) & ~7, M - 8) + (row & 7), gn = min(go, N - 8);
    if (gm < ((m0 + row) & ~7) || go >= N) continue;   // (the row or the whole octet belongs to its neighbour)
    uint16_t *dst = C + size_t(gm) * ldc + gn;
    const uint16_t *src = o + row * OP + (t % OCT) * 8;
    if (beta == 0.f || gn == go) __builtin_memcpy(dst, src, 16);
    else
      for (int e = go - gn; e < 8; ++e) dst[e] = src[e];
  }
}

template <bool BF16, bool AK, bool BKc>
void launch_tile(int bt, int ks, const uint16_t *A, int lda, const uint16_t *B, int ldb, uint16_t *C, int ldc, int M, int N, int K,
                 float alpha, float beta, hipStream_t s) {
  const unsigned ab = unsigned((size_t(AK ? M - 1 : K - 1) * lda + (AK ? K : M)) * 2);
  const unsigned bb = unsigned((size_t(BKc ? N - 1 : K - 1) * ldb + (BKc ? K : N)) * 2);
  const int mt = (M + bt - 1) / bt, tiles = mt * ((N + bt - 1) / bt);
  const dim3 grid(unsigned((tiles + 7) / 8 * 8));
#define SGH_TILE_CASE(BT_, KS_)                                                                                                     \
  hipLaunchKernelGGL((k_gemm16_tile<BF16, AK, BKc, BT_, KS_>), grid, dim3(256 * KS_), 0, s, A, lda, ab, B, ldb, bb, C, ldc, M, N,   \
                     K, mt, tiles, alpha, beta)
  if (bt == 128) SGH_TILE_CASE(128, 1);
  else if (ks == 2) SGH_TILE_CASE(64, 2);
  else SGH_TILE_CASE(64, 1);
#undef SGH_TILE_CASE
}

// The split kernel's tile and the wavefronts that share one, and whether it can take the problem at all.  16-wide tiles win while
// 32-wide ones leave half of the CUs without a workgroup (128 x 10 x 4096 NN 8.7 / 13.5 us); four wavefronts are enough for short
// reductions (784 x 1000 x 128: 5.0 / 5.1 us with 4 / 8), 16 gain nothing over 8 (512 x 1024 x 2048: 17.6 / 17.5).
bool split_plan(int M, int N, int K, int *tile, int *waves) {
  const long t32 = long((M + 31) / 32) * ((N + 31) / 32), cus = sgh_num_cus();
  if (t32 > 4 * cus) return false;
  *tile = 2 * t32 < cus ? 16 : 32;
  *waves = K < 256 ? 4 : 8;
  return (M + *tile - 1) / *tile <= 65535;
}

// Whether the tiled kernel is the better one where both can run.  The lines lie where the fewest of 1500 products lose to the other
// kernel (drawn over 8..4096 rows and columns, 8..8192 indices, all four layouts, replayed from a graph; us, split / tiled):
//   More than one 32-wide tile per CU: the tiled one, unless the reduction is short beside a launch (1024^3 NN 16.5 / 7.0, 512 x 1024 x
// 2048 NN 16.8 / 10.2; 504 x 904 x 104 NT 3.3 / 3.6, 44 x 5002 x 49 NT 3.0 / 3.7; with rows at odd elements 129 x 1648 x 587 TT 12.1 / 6.4).
//   Fewer: 64-wide tiles leave most of the CUs without a workgroup, and the split kernel is the better one however long the reduction is
// (256 x 1000 x 2048 NN 10.0 / 11.0, 472 x 54 x 5911 NN 21.1 / 30.3, 208 x 744 x 4304 NT 12.8 / 17.6, 974 x 36 x 6700 NN 13.4 / 29.1), except
// with rows at odd elements, where its loads take several times as long (780 x 213 x 4336 NN 82 / 26, 180 tiles x 2984 NN 2.6 times, 128 x 1657
// TT 1.8 times; but 54 tiles x 3323 NN 13.4 / 18.4, 25 x 1795 NT 0.8 times).  A transposed and B not, both walk along their rows and odd
// ones cost little (231 x 791 x 695 5.4 / 6.8, 1643 x 69 x 7633 36 / 43).
// 59 of the 1500 are more than 5 per cent from the better kernel, 0.6 per cent at the geometric mean.
bool tile_pays(bool ta, bool tb, int M, int N, int K, int lda, int ldb) {
  const long t32 = long((M + 31) / 32) * ((N + 31) / 32), cus = sgh_num_cus(), work = t32 * K;
  const bool odd = (lda | ldb) & 1;
  if (t32 > cus) return work > (odd ? 30000 : 100000);
  if (!odd || (ta && !tb)) return false;
  return !ta && !tb && (ldb & 1) ? work > 30000 : 4 * t32 >= cus && work > 100000;
}

// The tiled kernel's tile and groups.  128-wide tiles (half the loads per product) once they give every CU one and the reduction
// is long enough to matter (64 / 128: 2048 x 4096 x 1200 NT 46 / 30 us, 512 tiles; 700 x 6000 x 700 NT 18.5 / 17.7, 282; 1500^3 23.5 /
// 24.9, 144; 2232 x 2280 x 40 TN 6.4 / 7.1).  Two groups halve the chain of a workgroup that has its CU to itself (1024^3 8.4 / 7.0 with
// 256 tiles, 700 x 700 x 6000 39 / 31 with 121; 1813 x 597 x 964 11.8 / 12.1 with 290); four gain nothing more (6.9, 31.3).
// False where the workgroups are more than a launch holds (2^32 threads).
bool tile_plan(int M, int N, int K, int *bt, int *ks) {
  const long t64 = long((M + 63) / 64) * ((N + 63) / 64), t128 = long((M + 127) / 128) * ((N + 127) / 128), cus = sgh_num_cus();
  *bt = t128 > cus && K >= 256 ? 128 : 64;
  *ks = t64 <= cus && K > 2 * TK ? 2 : 1;
  return (*bt == 128 ? t128 : t64) <= (long(1) << 24) - 8;
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
  int tile, waves, bt, ks;
  const bool small = K > 0 && size_t(transA ? K : M) * lda < (size_t(1) << 30) &&
                     size_t(transB ? N : K) * ldb < (size_t(1) << 30);   // operands addressed with 32-bit byte offsets
  const bool split = small && split_plan(M, N, K, &tile, &waves), octets = M >= 8 && N >= 8 && K >= 8;
  if (small && octets && !(split && !tile_pays(transA, transB, M, N, K, lda, ldb)) && tile_plan(M, N, K, &bt, &ks)) {
    if (!transA && transB) launch_tile<BF16, true, true>(bt, ks, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else if (!transA) launch_tile<BF16, true, false>(bt, ks, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else if (transB) launch_tile<BF16, false, true>(bt, ks, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    else launch_tile<BF16, false, false>(bt, ks, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
    SGH_LAUNCH_CHECK();
    return SGH_OK;
  }
  if (split) {
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
