// fp32 data gradients of convolutions with at most four input channels, 3x3 and 5x5, stride 1 (the first layer of a small network):
//   dx[n][c][h][w] = sum_k sum_{r,s} dy[n][k][h + pad - r][w + pad - s] * W[k][c][r][s]
// On matrix tiles such a layer fills 4 of 32 rows; as one GEMM into columns and a gather (igemm.hip) it writes and reads a matrix of
// R * S times dx: 128 images of 3 channels of 32 x 32, 5x5 to 32 filters, 32 + 18 us.  Its products are few enough for the vector ALUs.
//   A workgroup of four or eight wavefronts owns 8 x 32 pixels of an image, all channels; wavefront v of n takes the filters v, v + n, ...: it stages
// its own 12 x 36 pixels of dy[n][k] in LDS (the next filter's on their way in registers, no barrier), a lane computes four neighbouring
// pixels of every channel, 300 products on 40 values from LDS, with the filter in scalar registers.  A filter's taps are summed on their
// own and added to the lane's sums with one rounding, and the wavefronts' sums are added in order.
// Bound by the vector ALUs and, where a CU has few workgroups, by the chain of a filter (LDS, scalar loads, 144 to 400 products: 0.6 to 1.1 us).
// That layer 43.8 -> 18.3 us, 67 x 1 x 30 x 36, 5x5 to 17 26.7 -> 8.2, 111 x 2 x 47 x 37, 3x3 to 191 74 -> 64; error 0.5 to 1.0 times.
// The data gradient has no padding in its definition: with an infinity or a NaN in the filter the taps that fall outside dy are left out
// one by one.
#include "common.h"

namespace {

constexpr int TH = 8, TW = 32;   // a lane: row lane / 8, columns 4 (lane % 8) .. + 3
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

struct Args {
  const float *dy, *W;
  float *dx;
  int K, P, Q, H, Wd, pad, bands, strips;   // bands of TH rows, strips of TW columns of an image
  unsigned dy_bytes;
};

template <int C, int R, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void k_dgrad_few(Args a) {
  constexpr int VR = TH + R - 1, VC = TW + R - 1, PITCH = (VC + 3) & ~3, E = (VR * VC + 63) / 64, RS = R * R;
  __shared__ __align__(16) float tiles[WAVES][VR * PITCH + 4];
  __shared__ float sums[WAVES - 1][C * 4][64];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int strip = int(blockIdx.x) % a.strips, rest = int(blockIdx.x) / a.strips, band = rest % a.bands, n = rest / a.bands;
  const int h0 = band * TH, w0 = strip * TW;
  const int p0 = h0 + a.pad - (R - 1), q0 = w0 + a.pad - (R - 1);   // dy position of the tile's first element
  const rsrc_t rdy = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.dy), 0, a.dy_bytes, 0x00020000);
  float *const tile = tiles[wave];
  int off[E], at[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = e * 64 + lane, vr = i / VC, vc = i - vr * VC, p = p0 + vr, q = q0 + vc;
    const bool ok = i < VR * VC && unsigned(p) < unsigned(a.P) && unsigned(q) < unsigned(a.Q);
    off[e] = ok ? ((n * a.K * a.P + p) * a.Q + q) * 4 : int(0x80000000u);
    at[e] = i < VR * VC ? vr * PITCH + vc : VR * PITCH;   // (the surplus lanes write beside the tile)
  }
  const int plane = a.P * a.Q * 4;
  float next[E];
  auto request = [&](int k) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      next[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rdy, k < a.K ? off[e] : int(0x80000000u), k * plane, 0));
  };
  f32x4 acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int row = lane >> 3, col = 4 * (lane & 7);
  request(wave);
  for (int k = wave; k < a.K; k += WAVES) {
#pragma unroll
    for (int e = 0; e < E; ++e) tile[at[e]] = next[e];
    request(k + WAVES);
    const float *w = a.W + size_t(k) * C * RS;   // (uniform)
    // x * 0 is not zero for an infinity or a NaN
    float zero = 0.f;
#pragma unroll
    for (int i = 0; i < (C * RS + 63) / 64; ++i)
      if (i * 64 + lane < C * RS) zero = fmaf(w[i * 64 + lane], 0.f, zero);
    const bool odd = __any(!(zero == 0.f));
    f32x4 s[C];
#pragma unroll
    for (int c = 0; c < C; ++c) s[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!odd) {
#pragma unroll
      for (int vr = 0; vr < R; ++vr) {   // tap r = R - 1 - vr reads row `row + vr` of the tile
        float v[4 + ((R + 2) & ~3)];
#pragma unroll
        for (int u = 0; u < int(sizeof(v) / 16); ++u) {
          const f32x4 q = *reinterpret_cast<const f32x4 *>(tile + (row + vr) * PITCH + col + 4 * u);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * u + e] = q[e];
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int vc = 0; vc < R; ++vc) {
            const float f = w[c * RS + (R - 1 - vr) * R + (R - 1 - vc)];
#pragma unroll
            for (int e = 0; e < 4; ++e) s[c][e] = fmaf(f, v[vc + e], s[c][e]);
          }
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < RS; ++i) {
        const int vr = i / R, vc = i - vr * R, p = p0 + row + vr;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int q = q0 + col + vc + e;
          if (unsigned(p) < unsigned(a.P) && unsigned(q) < unsigned(a.Q)) {
            const float v = tile[(row + vr) * PITCH + col + vc + e];
#pragma unroll
            for (int c = 0; c < C; ++c) s[c][e] = fmaf(w[c * RS + RS - 1 - i], v, s[c][e]);
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[c][e] += s[c][e];
  }
  if (wave > 0)
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) sums[wave - 1][c * 4 + e][lane] = acc[c][e];
  __syncthreads();
  if (wave > 0 || h0 + row >= a.H) return;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    float *out = a.dx + ((size_t(n) * C + c) * a.H + h0 + row) * a.Wd + w0 + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = acc[c][e];
#pragma unroll
      for (int w = 0; w < WAVES - 1; ++w) v += sums[w][c * 4 + e][lane];
      if (w0 + col + e < a.Wd) out[e] = v;
    }
  }
}

}  // namespace

// Up to 64 filters: the columns' reduction runs on the matrix instructions, here a wavefront walks its share of the filters one by one.  Beyond,
// few images are slower on four wavefronts: 1 x 3 x 61 x 77, 5x5 to 79 23.0 / 26.5, 3 x 4 x 32 x 30 to 167 22.9 / 35.3, 13 x 4 x 32 x 22 to 964
// 84 / 222.
bool sgh_dgrad_few_supported(const sgh_conv_geom *g) {
  const size_t lim = size_t(1) << 31, wgs = size_t(g->N) * ((g->H + TH - 1) / TH) * ((g->W + TW - 1) / TW);
  return wgs < size_t(1) << 24 &&   // (a launch holds less than 2^32 threads)
         g->C <= 4 && g->K <= 64 && g->R == g->S && (g->R == 3 || g->R == 5) && g->stride_h == 1 && g->stride_w == 1 && g->pad_h == g->pad_w &&
         g->pad_h < g->R && size_t(g->N) * g->K * g->P * g->Q * 4 < lim && size_t(g->N) * g->C * g->H * g->W * 4 < lim;
}

int sgh_dgrad_few_run(const sgh_conv_geom *g, const float *dy, const float *W, float *dx, hipStream_t s) {
  Args a{dy, W, dx, g->K, g->P, g->Q, g->H, g->W, g->pad_h, (g->H + TH - 1) / TH, (g->W + TW - 1) / TW,
         unsigned(size_t(g->N) * g->K * g->P * g->Q * 4)};
  const dim3 grid(unsigned(g->N) * unsigned(a.bands) * unsigned(a.strips));
  sgh_prof_kernel_scope prof("conv_dgrad/k_dgrad_few", 2.0 * g->N * g->K * g->P * g->Q * double(g->C) * g->R * g->S, s);
  const long wgs = long(grid.x), cus = sgh_num_cus();
  // Eight wavefronts halve the chain of a workgroup that has its CU to itself, or shares it with one or two: us in columns / on four / eight, 5x5,
  // 2 x 4 x 16 x 13 to 64 (bfloat16) 27.5 / 34.5 / 25.6, 5 x 4 x 21 x 21 to 61 21.1 / 23.9 / 19.4, 16 x 4 x 17 x 17 to 63 30.3 / 35.2 / 27.4; with
  // four, 73 of 500 layers of 40 to 64 filters were slower than in columns.  Beyond, the vector ALUs are busy either way (15 x 4 x 57 x 78, 3x3 to
  // 10 5.9 / 6.7, 13 x 3 x 96 x 112 to 44 16.3 / 17.6), and beside another stream's kernels four leave those more room (the small CNN's step, 512
  // workgroups, 32 filters: alone 16.2 / 15.3, the step 278.6 / 280.2).
  const bool eight = (wgs <= cus && g->K > 8) || (wgs <= (g->R == 5 ? 3 : 2) * cus && g->K > 32);
#define SGH_FEW_KERNEL(C_, R_)                                                             \
  do {                                                                                     \
    if (eight) SGH_LAUNCH_TIMED((k_dgrad_few<C_, R_, 8>), grid, dim3(512), 0, s, a);       \
    else SGH_LAUNCH_TIMED((k_dgrad_few<C_, R_, 4>), grid, dim3(256), 0, s, a);             \
  } while (0)
#define SGH_FEW(C_)                  \
  if (g->R == 3) SGH_FEW_KERNEL(C_, 3); \
  else SGH_FEW_KERNEL(C_, 5)
  switch (g->C) {
    case 1: SGH_FEW(1); break;
    case 2: SGH_FEW(2); break;
    case 3: SGH_FEW(3); break;
    default: SGH_FEW(4); break;
  }
#undef SGH_FEW
#undef SGH_FEW_KERNEL
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}
