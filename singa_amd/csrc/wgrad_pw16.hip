// Weight gradients of 1x1 / stride 1 / unpadded convolutions on 16-bit NCHW tensors:
//   dW[k][c] = sum over images and pixels of dy[n][k][pix] * x[n][c][pix]      (v_mfma_f32_32x32x16_{f16,bf16}, fp32 sums)
// Both operands have the reduction index contiguous, so a tile of either is staged as it lies in memory, [channel][64 pixels], and
// its 16-byte reads are the fragments.  A chunk of the reduction is eight octets of pixels; a plane's last octet ends with the plane,
// and the pixels that it shares with the one before are cleared in both operands.
// A workgroup owns a BM x BN tile of dW and a part of the chunks: two groups of four wavefronts (a wavefront a quarter of the tile)
// take alternate chunks through two register sets (requested two chunks ahead) and two LDS buffers, one barrier per chunk, and their
// sums are added in order.  Partial images of the parts are added in order by the caller; one part is rounded and stored at once.
//   Bound by bytes on planes of 56 x 56; on small ones by what a CU draws from L2 (16 bytes per cycle, as in the other kernels of this
// family), on short reductions by the launch, one chain of loads and the partial images: as few parts as fill the CUs.  Requests
// placed ahead of the products instead of behind them (the compiler's order) were no faster.
#include <atomic>
#include <type_traits>

#include "common.h"
#include "fastdiv.h"
#include "storage.h"
#include "wgrad_pw16.h"

namespace {

constexpr int TK = 64, KS = 2, kOOB = int(0x80000000u);

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

struct Args {
  const uint16_t *dy, *x;
  float *partial;     // [parts][K][C], or null: dW
  uint16_t *dW;
  int K, C, HW, QO, over;   // octets of a plane; pixels that its last one shares with the one before
  int octets, mtiles, tiles, parts, chunks, per_part;
  unsigned dy_bytes, x_bytes;
  sgh_fastdiv d_qo;
};

template <bool BF16>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Rows row0 .. row0 + B of one operand: thread t (of 256) loads octet t % 8 of rows 32 j + t / 8
template <int B>
struct Panel {
  static constexpr int N = B / 32;
  rsrc_t r;
  int off[N];   // of the row, in bytes; out of range when it does not exist
  int image;    // bytes of one image
  u32x4 v[2][N];
  __device__ __forceinline__ void init(const uint16_t *p, unsigned bytes, int row0, int rows, int HW) {
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p), 0, bytes, 0x00020000);
    image = rows * HW * 2;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int row = row0 + 32 * j + int((threadIdx.x & 255) >> 3);
      off[j] = row < rows ? row * HW * 2 : kOOB;
    }
  }
  template <int S>
  __device__ __forceinline__ void request(int n, int pixel, bool there) {
    const int base = n * image + pixel * 2;
#pragma unroll
    for (int j = 0; j < N; ++j)   // (a row that does not exist: 2^31 + base, still out of range)
      v[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, there ? int(unsigned(off[j]) + unsigned(base)) : kOOB, 0, 0));
  }
  template <int S>
  __device__ __forceinline__ void stage(uint16_t *tile, u32x4 keep, bool masked) {
    const int t = threadIdx.x & 255;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int row = 32 * j + (t >> 3);
      *reinterpret_cast<u32x4 *>(tile + row * TK + (((t & 7) ^ ((row >> 1) & 7)) * 8)) = masked ? v[S][j] & keep : v[S][j];
    }
  }
  static __device__ __forceinline__ u32x4 fragment(const uint16_t *tile, int tile32, int step) {
    const int lane = threadIdx.x & 63, row = 32 * tile32 + (lane & 31);
    return *reinterpret_cast<const u32x4 *>(tile + row * TK + (((2 * step + (lane >> 5)) ^ ((row >> 1) & 7)) * 8));
  }
};

template <bool BF16, int BM, int BN>
__global__ __launch_bounds__(256 * KS) void k_wgrad_pw16(Args a) {
  constexpr int TM = BM / 64, TN = BN / 64, HALF = (BM + BN) * TK;
  extern __shared__ __align__(16) uint16_t lds_pw[];
  // workgroup w runs on XCD w % 8: the tiles of one part read the same pixels through one L2, or, with fewer than eight parts, through the L2s
  // of neighbouring XCDs (in the order of the workgroups all eight read all of them: 10 x 856 x 62 x 54 -> 288, 35 tiles in seven parts,
  // 70 us, the 77 MB eight times, 47 now; 110 x 566 x 16 x 15 -> 413, four parts, 58 -> 42)
  int tile, part;
  const int slot = int(blockIdx.x) >> 3, xcd = int(blockIdx.x) & 7;
  if ((a.parts & 7) == 0) {
    tile = slot % a.tiles, part = (slot / a.tiles) * 8 + xcd;
  } else {
    const int total = a.tiles * a.parts, per = (total + 7) >> 3, l = xcd * per + slot;
    if (l >= total) return;
    tile = l % a.tiles, part = l / a.tiles;
  }
  const int m0 = (tile % a.mtiles) * BM, n0 = (tile / a.mtiles) * BN;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = (wave >> 1) & 1, wn = wave & 1;
  const int group = wave >> 2;
  uint16_t *const lds0 = lds_pw + group * 2 * HALF;
  const int c_begin = part * a.per_part, c_end = min(a.chunks, c_begin + a.per_part);
  Panel<BM> pa;
  Panel<BN> pb;
  pa.init(a.dy, a.dy_bytes, m0, a.K, a.HW);
  pb.init(a.x, a.x_bytes, n0, a.C, a.HW);
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  int cut[2];   // elements to clear at the front of the octet of either register set
  auto request = [&](auto SET, int c) {
    constexpr int S = decltype(SET)::value;
    const int chunk = c_begin + c * KS + group, o = chunk * 8 + (t & 7), n = a.d_qo.div(o), p = o - n * a.QO;
    const bool there = chunk < c_end && o < a.octets;
    const int pixel = min(8 * p, a.HW - 8);
    cut[S] = 8 * p - pixel;
    pa.template request<S>(n, pixel, there);
    pb.template request<S>(n, pixel, there);
  };
  auto stage = [&](auto SET) {
    constexpr int S = decltype(SET)::value;
    u32x4 keep = {~0u, ~0u, ~0u, ~0u};
    if (a.over) {
#pragma unroll
      for (int i = 0; i < 4; ++i) keep[i] = cut[S] >= 2 * i + 2 ? 0u : cut[S] == 2 * i + 1 ? 0xffff0000u : ~0u;
    }
    pa.template stage<S>(lds0 + S * HALF, keep, a.over != 0);
    pb.template stage<S>(lds0 + S * HALF + BM * TK, keep, a.over != 0);
  };
  auto multiply = [&](const uint16_t *st) {
#pragma unroll
    for (int step = 0; step < TK / 16; ++step) {
      u32x4 fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = Panel<BM>::fragment(st, wm * TM + i, step);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j] = Panel<BN>::fragment(st + BM * TK, wn * TN + j, step);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma<BF16>(fa[i], fb[j], acc[i][j]);
    }
  };
  const int rounds = (c_end - c_begin + KS - 1) / KS;
  typedef std::integral_constant<int, 0> Set0;
  typedef std::integral_constant<int, 1> Set1;
  auto step = [&](auto SET, int c) {   // chunk c of the group; false at the end
    constexpr int S = decltype(SET)::value;
    __syncthreads();
    request(SET, c + 2);
    multiply(lds0 + S * HALF);
    if (c + 1 >= rounds) return false;
    stage(std::integral_constant<int, S ^ 1>{});
    return true;
  };
  request(Set0{}, 0);
  request(Set1{}, 1);
  stage(Set0{});
  for (int c = 0; step(Set0{}, c) && step(Set1{}, c + 1); c += 2) {
  }
  {   // the groups' sums in their order
    __syncthreads();
    float *const mine = reinterpret_cast<float *>(lds_pw + group * 2 * HALF) + (wave & 3) * (TM * TN * 1024);
    if (group > 0)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) mine[((i * TN + j) * 16 + v) * 64 + lane] = acc[i][j][v];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g) {
      const float *other = reinterpret_cast<const float *>(lds_pw + g * 2 * HALF) + (wave & 3) * (TM * TN * 1024);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] += other[((i * TN + j) * 16 + v) * 64 + lane];
    }
  }
  float *const out = a.partial ? a.partial + size_t(part) * a.K * a.C : nullptr;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + (wn * TN + j) * 32 + (lane & 31);
    if (col >= a.C) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = m0 + (wm * TM + i) * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row >= a.K) continue;
        if (out) out[size_t(row) * a.C + col] = acc[i][j][v];
        else a.dW[size_t(row) * a.C + col] = BF16 ? sgh_f32_to_bf16(acc[i][j][v]) : sgh_f32_to_f16(acc[i][j][v]);
      }
  }
}

template <bool BF16, int BM, int BN>
int launch(const Args &a, hipStream_t s) {
  auto kern = k_wgrad_pw16<BF16, BM, BN>;
  constexpr size_t bytes = size_t(KS) * 2 * (BM + BN) * TK * 2;
  static_assert(size_t(BM) * BN * 4 <= bytes / KS, "a group's sums in its buffers");
  static std::atomic<bool> allowed{false};
  if (!allowed.load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)) != hipSuccess)
      return SGH_EUNSUPPORTED;
    allowed.store(true, std::memory_order_relaxed);
  }
  SGH_LAUNCH_TIMED(kern, dim3((unsigned(a.tiles) * unsigned(a.parts) + 7) / 8 * 8), dim3(256 * KS), bytes, s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

template <bool BF16>
int launch_plan(const Args &a, const sgh_wgrad_pw16_plan &p, hipStream_t s) {
  if (p.bm == 128) return p.bn == 128 ? launch<BF16, 128, 128>(a, s) : launch<BF16, 128, 64>(a, s);
  return p.bn == 128 ? launch<BF16, 64, 128>(a, s) : launch<BF16, 64, 64>(a, s);
}

}  // namespace

// The tile and the parts with the least expected time.  The constants (us: a launch, a round of a workgroup on its CU, the partial images written
// and summed) are fitted to 2400 timings, 200 layers drawn over 1..128 images, 3..1024 channels, planes of 7..112, to 8 per cent; the choice is
// 1.7 per cent from the best of the twelve that were timed.  bfloat16 with the sum of the parts, k_wgrad16 / here, us:
//   21 x 64 x 48 x 48 -> 256 19.9 / 12.3, 21 x 128 x 24 x 24 -> 512 17.8 / 11.0, 21 x 512 x 6 x 6 -> 2048 22.3 / 8.2;
//   128 x 64 x 56 x 56 -> 256 53 / 42.5 (6.0 TB/s), 128 x 512 x 28 x 28 -> 128 35.5 / 32.8, 128 x 256 x 14 x 14 -> 1024 35.8 / 35.0.
// Planes of an odd number of pixels leave rows at odd elements, where a 16-byte load takes twice the lines: from about 25 us on k_wgrad16,
// with twice the wavefronts, is faster there (128 x 512 x 7 x 7 -> 2048 42.4 / 46.1, 59 x 964 x 21 x 21 -> 835 93 / 123; 8 x 592 x 29 x 33 ->
// 575 28.8 / 31.0).
sgh_wgrad_pw16_plan sgh_wgrad_pw16_plan_of(const sgh_conv_geom *g) {
  sgh_wgrad_pw16_plan p{};
  if (g->R != 1 || g->S != 1 || g->stride_h != 1 || g->stride_w != 1 || g->pad_h != 0 || g->pad_w != 0 || g->H * g->W < 8) return p;
  const size_t lim = size_t(1) << 30, HW = size_t(g->H) * g->W;   // byte offsets into x and dy stay below 2^31
  if (size_t(g->N) * g->C * HW >= lim || size_t(g->N) * g->K * HW >= lim || size_t(g->K) * g->C >= lim) return p;
  p.chunks = int((size_t(g->N) * ((HW + 7) / 8) + 7) / 8);
  const int cus = sgh_num_cus();
  double best = -1;
  for (int shape = 0; shape < 4; ++shape)
    for (int half = 1; half <= 4; half *= 2) {   // workgroups wanted, in halves of the CUs
      const int bm = shape & 1 ? 128 : 64, bn = shape & 2 ? 128 : 64;
      if ((bm == 128 && g->K <= 64) || (bn == 128 && g->C <= 64)) continue;
      const long tiles = long((g->K + bm - 1) / bm) * ((g->C + bn - 1) / bn);
      if (tiles >= (1l << 30)) continue;
      long parts = half * cus / 2 / tiles;
      if (parts > p.chunks / KS) parts = p.chunks / KS;
      if (parts < 1) parts = 1;
      if (parts >= 8) parts &= ~7l;   // (every XCD whole parts; the last of them may then be short or empty)
      const int per_part = int((p.chunks + parts - 1) / parts);
      if (parts < 8) parts = (p.chunks + per_part - 1) / per_part;
      const int rounds = (per_part + KS - 1) / KS;
      const double wgs = double(tiles) * parts, at_once = shape == 0 ? 2.0 * cus : cus;   // (LDS: two of the small tiles on a CU)
      const double turns = wgs <= at_once ? 1 : double((tiles * parts + long(at_once) - 1) / long(at_once));
      const double round = shape == 3 ? 1.15 : shape ? 0.91 : wgs <= cus ? 0.53 : 0.52 * (wgs < at_once ? wgs / cus : 2);
      double us = 4.2 + turns * rounds * round * (HW % 2 ? 1.28 : HW % 64 ? 1.06 : 1);
      if (parts > 1) us += 2.3 + double(parts) * g->K * g->C * 3.4e-6;
      if (best >= 0 && us >= best) continue;
      best = us;
      p.bm = bm, p.bn = bn, p.tiles = int(tiles), p.parts = int(parts), p.per_part = per_part;
    }
  p.ok = HW % 2 == 0 || best <= 25;
  return p;
}

int sgh_wgrad_pw16_run(const sgh_conv_geom *g, const sgh_wgrad_pw16_plan &p, const uint16_t *dy, const uint16_t *x, float *partial,
                       uint16_t *dW, bool bf16, hipStream_t s) {
  Args a;
  a.dy = dy, a.x = x, a.partial = p.parts > 1 ? partial : nullptr, a.dW = dW;
  a.K = g->K, a.C = g->C, a.HW = g->H * g->W, a.QO = (a.HW + 7) / 8, a.over = 8 * a.QO - a.HW;
  a.octets = g->N * a.QO, a.mtiles = (g->K + p.bm - 1) / p.bm, a.tiles = p.tiles, a.parts = p.parts;
  a.chunks = p.chunks, a.per_part = p.per_part, a.d_qo = sgh_fastdiv(a.QO);
  a.dy_bytes = unsigned(size_t(g->N) * g->K * a.HW * 2), a.x_bytes = unsigned(size_t(g->N) * g->C * a.HW * 2);
  return bf16 ? launch_plan<true>(a, p, s) : launch_plan<false>(a, p, s);
}
