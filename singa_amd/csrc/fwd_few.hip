// fp32 forward convolution over fewer than eight input channels, 3x3, 5x5 or 7x7 at any stride and padding (GpuConvForward,
// src/model/operation/convolution.cc:585-620): the first layer of a network whose geometry is not the residual stem's.
//
// The generic kernel pads the channels of every tap to its reduction chunk of 16; here the reduction runs over (channel, window
// row, window column), the columns padded to an even number, two indices per v_mfma_f32_32x32x2_f32:
//
//   * a workgroup (four wavefronts) takes `rows` whole output rows of the flattened (image, row) index, up to 256 pixels, and
//     32 or 64 filters; a wavefront takes every fourth block of 32 pixels, filters are the matrix rows;
//   * the input rows under them sit in LDS in a "virtual" row space in which every image owns P * stride + R - 1 rows, so that a
//     tile may cross images and the padding is zeros; the window of a pixel is an offset of the step alone;
//   * the filters are written to LDS as [channel, row, column][filter], zero in the padding column; the pixel that it meets is
//     replaced by zero, so that an infinity beside a window does not become a NaN inside it.
//
// 128 images of 3 channels, 32 x 32, to 32 filters 5x5: 92 -> 26 us; 90 drawn layers 2.2 times as fast, the slowest 1.1, with the
// same error against float64.  Half of it is the staging of a tile, which nothing overlaps but the other workgroups of the CU.
#include <type_traits>

#include "common.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int NT = 256, kPixels = 256;

struct FfArgs {
  const float *x, *W, *bias;
  float *y;
  int N, C, H, Wd, K, P, Q, R, stride, pad_h, pad_w;
  int rows, pitch, srows;   // output rows of a tile, columns and rows of the slab
};

template <int S, int KB>
__global__ __launch_bounds__(NT) void k_fwd_few(FfArgs a) {
  constexpr int SE = S + 1, KP = KB + 1, MB = KB / 32, NB = kPixels / 32 / (NT / 64);
  extern __shared__ __align__(16) float lds[];
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int crs = a.C * a.R * SE;
  float *const ws = lds, *const xs = lds + crs * KP;   // [crs][KP], [C][srows][pitch]
  const int k0 = int(blockIdx.y) * KB, row0 = int(blockIdx.x) * a.rows, VH = a.P * a.stride + a.R - 1;
  const int n0 = row0 / a.P, vbase = n0 * VH + (row0 - n0 * a.P) * a.stride;

  // filters in the order of memory (LDS rows of KB + 1: a column of them falls into as many banks), four requests in flight
  const int CRS = a.C * a.R * S, live = min(KB, a.K - k0) * CRS;
  const float *const W = a.W + size_t(k0) * CRS;
  for (int i0 = t; i0 < KB * CRS; i0 += 4 * NT) {
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = i0 + u * NT < live ? W[i0 + u * NT] : 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * NT, k = i / CRS, e = i - k * CRS;
      if (i < KB * CRS) ws[(e / S * SE + e % S) * KP + k] = v[u];
    }
  }
  for (int i = t; i < a.C * a.R * KB; i += NT) ws[(i / KB * SE + S) * KP + i % KB] = 0.f;
  const int xelems = a.C * a.srows * a.pitch;
  for (int i0 = t; i0 < xelems; i0 += 4 * NT) {
    float d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * NT, cr = i / a.pitch, col = i - cr * a.pitch, c = cr / a.srows, v = vbase + cr - c * a.srows, n = v / VH;
      const int h = v - n * VH - a.pad_h, w = col - a.pad_w;
      const bool in = i < xelems && n < a.N && unsigned(h) < unsigned(a.H) && unsigned(w) < unsigned(a.Wd);
      d[u] = in ? a.x[((size_t(n) * a.C + c) * a.H + h) * a.Wd + w] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * NT < xelems) xs[i0 + u * NT] = d[u];
  }

  // this lane's pixels (columns of the B operand); those beyond the tile repeat its first one and are not stored
  const int pixels = min(a.rows, a.N * a.P - row0) * a.Q;
  int boff[NB];
  size_t out[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int pix = (j * (NT / 64) + wave) * 32 + l32, at = pix < pixels ? pix : 0;
    const int r = at / a.Q, q = at - r * a.Q, n = (row0 + r) / a.P, p = row0 + r - n * a.P;
    boff[j] = (n * VH + p * a.stride - vbase) * a.pitch + q * a.stride + half;
    out[j] = (size_t(n) * a.K * a.P + p) * a.Q + q;
  }
  v16f acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  __syncthreads();

  auto multiply = [&](auto blocks) {   // this wavefront's first blocks of pixels
    const float *ap = ws + half * KP + l32;
    for (int c = 0; c < a.C; ++c)
      for (int r = 0; r < a.R; ++r, ap += SE * KP) {
        const float *bp = xs + (c * a.srows + r) * a.pitch;
#pragma unroll
        for (int s = 0; s < SE; s += 2) {
          float w[MB];
#pragma unroll
          for (int i = 0; i < MB; ++i) w[i] = ap[s * KP + 32 * i];
#pragma unroll
          for (int j = 0; j < blocks; ++j) {
            float v = bp[boff[j] + s];
            if (s + 1 >= S) v = half ? 0.f : v;
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[i], v, acc[i][j], 0, 0, 0);
          }
        }
      }
  };
  static_assert(NB == 2, "");
  if ((NT / 64 + wave) * 32 < pixels) multiply(std::integral_constant<int, 2>{});
  else if (wave * 32 < pixels) multiply(std::integral_constant<int, 1>{});

#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if ((j * (NT / 64) + wave) * 32 + l32 >= pixels) continue;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int k = k0 + 32 * i + 8 * (v >> 2) + 4 * half + (v & 3);
        if (k < a.K) a.y[out[j] + size_t(k) * a.P * a.Q] = acc[i][j][v] + (a.bias ? a.bias[k] : 0.f);
      }
  }
}

struct FfPlan {
  bool ok;
  int kb, rows, pitch, srows;
  size_t lds;
};

FfPlan plan(const sgh_conv_geom *g) {
  FfPlan p{};
  if (sgh_env().fwd_fewc_off || g->groups > 1 || g->C < 1 || g->C >= 8 || g->R != g->S || (g->R != 3 && g->R != 5 && g->R != 7)) return p;
  if (g->stride_h != g->stride_w || g->Q > kPixels || g->P < 1 || g->Q < 1) return p;
  const size_t lim = size_t(1) << 31;
  const size_t vh = size_t(g->P) * g->stride_h + g->R - 1;
  if (size_t(g->N) * vh >= lim / 4 || size_t(g->N) * g->P >= lim / 4) return p;
  const int se = (g->S + 1) & ~1;
  // 64 filters, 32 where that would leave CUs without a tile (one image of 7 channels, 91 x 101, to 84 filters 3x3:
  // 18 us on 64, 16 on 32);
  // 256 pixels, fewer for the same reason
  const long total = long(g->N) * g->P, tiles = (total * g->Q + kPixels - 1) / kPixels;
  p.kb = g->K > 32 && tiles * ((g->K + 63) / 64) >= sgh_num_cus() ? 64 : 32;
  const long ktiles = (g->K + p.kb - 1) / p.kb;
  if (ktiles > 65535) return p;
  long rows = kPixels / g->Q;
  const long even = (total * ktiles + sgh_num_cus() - 1) / sgh_num_cus();
  if (rows > even) rows = even;
  p.rows = int(rows < 1 ? 1 : rows);
  p.pitch = (g->Q - 1) * g->stride_w + se;
  // (virtual rows: those of the tile and the rows between the images that it crosses)
  p.srows = p.rows * g->stride_h + (g->R - 1) * ((p.rows - 1) / g->P + 2);
  p.lds = (size_t(g->C) * g->R * se * (p.kb + 1) + size_t(g->C) * p.srows * p.pitch) * sizeof(float);
  p.ok = p.lds <= 160 * 1024;
  return p;
}

template <int S, int KB>
int launch(const FfArgs &a, const FfPlan &p, hipStream_t s) {
  auto kern = k_fwd_few<S, KB>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) !=
        hipSuccess)
      return SGH_EUNSUPPORTED;
    attr_set = true;
  }
  const long total = long(a.N) * a.P;
  SGH_LAUNCH_TIMED(kern, dim3(unsigned((total + p.rows - 1) / p.rows), unsigned((a.K + KB - 1) / KB)), dim3(NT), p.lds, s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

}  // namespace

int sgh_fwd_few_run(const sgh_conv_geom *g, const float *x, const float *W, const float *bias, float *y, hipStream_t s) {
  const FfPlan p = plan(g);
  if (!p.ok) return SGH_EUNSUPPORTED;
  const FfArgs a{x, W, bias, y, g->N, g->C, g->H, g->W, g->K, g->P, g->Q, g->R, g->stride_h, g->pad_h, g->pad_w, p.rows, p.pitch, p.srows};
  sgh_prof_scope prof("conv_fwd/k_fwd_few", 2.0 * g->N * g->K * g->P * g->Q * g->C * g->R * g->S, s);
  if (p.kb == 64) return g->S == 3 ? launch<3, 64>(a, p, s) : g->S == 5 ? launch<5, 64>(a, p, s) : launch<7, 64>(a, p, s);
  return g->S == 3 ? launch<3, 32>(a, p, s) : g->S == 5 ? launch<5, 32>(a, p, s) : launch<7, 32>(a, p, s);
}
