// Grouped convolutions with few channels per group (depthwise layers above all), directly on the vector ALUs.
//
// Such a layer moves far more bytes than it computes (a depthwise 3x3 has nine products per output), and a matrix tile
// would be almost empty, so the three passes are bound by reading and writing the tensors once -- and, run as one dense
// convolution per group, by their launches: 32 x 96 x 28 x 28 depthwise 3x3 took 1152 launches and 5.1 ms for the three
// passes; 27 us here (traced: forward and data gradient 8 us each, weight gradient 10 + 3.5; they overlap at the ends).
//
// Forward pass and data gradient are one kernel.  A "unit" is one group of one image; the channels of consecutive units
// are consecutive in memory.  A workgroup takes UB units x TP output rows: their source rows go into LDS as a zero-padded
// image (for the data gradient of a strided layer with zeros between the rows and columns, which makes it a stride-1
// correlation with the reversed filter), the filters beside them, and a thread computes strips of four output rows in
// one column, so that a row of the image is read once for all the outputs of the strip it contributes to.
//
// Weight gradient: a workgroup takes one (filter, input channel) pair and a chunk of the images, keeps the R x S sums
// in registers and adds them over its threads; the chunks' sums are added in chunk order by a second kernel, so results
// are the same on every run.
#include "common.h"
#include "fastdiv.h"
#include "storage.h"

namespace {

constexpr int GT = 256, STRIP = 4;
// Most channels per group, on either side, that take these kernels.  Against a dense convolution per group: 1 to 8 channels
// 17 times as fast (500 shapes, none slower); 9 to 16 still 8 times, but weight gradients of large planes in 16 bits, where the
// matrix instructions do the work of a few groups, down to 0.36 (23 x 56 x 83 x 92, four groups: 103 -> 288 us).
constexpr int kNarrow = 8;
// LDS per workgroup: six fit on a CU.  Over 240 shapes 48 KB take 1.14 times the time (0.80 to 3.07), 12 KB 0.90 (0.48 to 1.49).
constexpr int kLdsTarget = 24 * 1024;
constexpr int kLdsMost = 64 * 1024;

typedef __amdgpu_buffer_rsrc_t rsrc_t;

struct GroupArgs {
  int units, G;                 // N * G; groups
  int cs, cd;                   // channels per group of the source and of the destination
  int SH, SW, DH, DW;
  int dil, padh, padw;          // source element (y, x) sits at row y * dil + padh of the virtual image
  int TP, VR, VC;               // output rows per tile; rows and columns of the virtual image in LDS
  int UB;                       // units per workgroup
  int QN;                       // groups of four columns of the image that the tile reads; 0: narrow or dilated ones, value by value
  bool flip;                    // data gradient: reversed taps, filters indexed [source][destination]
  unsigned src_bytes;
  sgh_fastdiv d_vc, d_qn, d_vr, d_cs, d_dw, d_strips, d_cd, d_dil, d_G, d_taps;
};

template <class S>
__device__ __forceinline__ float ld_elem(rsrc_t r, int elem, bool ok) {
  typedef typename S::elem E;
  const int off = ok ? elem * int(sizeof(E)) : int(0x80000000u);
  if constexpr (sizeof(E) == 4) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else {
    const E e = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
    return S::ld(&e);
  }
}

template <class S>
__device__ __forceinline__ void ld_quad(rsrc_t r, int elem, bool ok, float (&v)[4]) {   // four elements, at any element's address
  typedef typename S::elem E;
  const int off = ok ? elem * int(sizeof(E)) : int(0x80000000u);
  if constexpr (sizeof(E) == 4) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4 w = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = w[e];
  } else {
    const auto w = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const E h = E(w[e >> 1] >> (16 * (e & 1)));
      v[e] = S::ld(&h);
    }
  }
}

template <class S>
__device__ __forceinline__ rsrc_t buffer_of(const typename S::elem *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<typename S::elem *>(p), 0, bytes, 0x00020000);
}

// Source rows of `planes` consecutive planes (first plane `plane0`, those from `planes_end` on are zero) into LDS as
// [plane][VR][VC]; row 0 of the virtual image is virtual row `vrow0`.  Returns whether this thread met an infinity or a NaN.
// (QUADS: loads of four columns in flight, 0 if a.QN is never set)
template <class S, int QUADS>
__device__ __forceinline__ bool stage_planes(float *lds, const GroupArgs &a, rsrc_t src, int plane0, int planes, int plane_step,
                                             int planes_end, int vrow0) {
  float zero = 0.f;   // until it has been multiplied with an infinity or a NaN
  if constexpr (QUADS > 0) if (a.QN) {
    constexpr int U = QUADS;
    // four columns per load (the last four of a row overlap the ones before): 2 700 values of three 28 x 28 planes are one round
    // of loads, where one value per load and two divisions each were three (depthwise 3x3 on
    // 32 x 96 x 28 x 28: 9.4 -> 8.0 us a pass)
    const int total = planes * a.VR * a.QN;
    for (int i0 = threadIdx.x; i0 < total; i0 += GT * U) {
      float v[U][4];
      int at[U], left[U];   // LDS index of the first column; columns of the image from there on
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * GT;
        const int row = a.d_qn.div(i), x = min(4 * (i - row * a.QN), a.SW - 4);
        const int pl = a.d_vr.div(row), y = vrow0 + row - pl * a.VR - a.padh;
        at[u] = row * a.VC + a.padw + x;
        left[u] = i < total ? a.VC - a.padw - x : 0;
        ld_quad<S>(src, ((plane0 + pl * plane_step) * a.SH + y) * a.SW + x, i < total && y >= 0 && y < a.SH && pl < planes_end, v[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (e < left[u]) {
            zero = fmaf(v[u][e], 0.f, zero);
            lds[at[u] + e] = v[u][e];
          }
        }
    }
    const int rows = planes * a.VR, right = a.VC - a.padw - a.SW;   // the columns beside the image
    for (int row = threadIdx.x; row < rows; row += GT) {
      for (int j = 0; j < a.padw; ++j) lds[row * a.VC + j] = 0.f;
      for (int j = 0; j < right; ++j) lds[row * a.VC + a.padw + a.SW + j] = 0.f;
    }
    return zero != 0.f;
  }
  constexpr int U = 4;
  const int total = planes * a.VR * a.VC;
  for (int i0 = threadIdx.x; i0 < total; i0 += GT * U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * GT;
      const int row = a.d_vc.div(i), j = i - row * a.VC;
      const int pl = a.d_vr.div(row), vr = row - pl * a.VR;
      const int yy = vrow0 + vr - a.padh, xx = j - a.padw;
      int y = yy, x = xx;
      bool ok = i < total && yy >= 0 && xx >= 0 && pl < planes_end;
      if (a.dil > 1) {
        y = a.d_dil.div(yy < 0 ? 0 : yy), x = a.d_dil.div(xx < 0 ? 0 : xx);
        ok = ok && y * a.dil == yy && x * a.dil == xx;
      }
      ok = ok && y < a.SH && x < a.SW;
      v[u] = ld_elem<S>(src, ((plane0 + pl * plane_step) * a.SH + y) * a.SW + x, ok);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      zero = fmaf(v[u], 0.f, zero);
      if (i0 + u * GT < total) lds[i0 + u * GT] = v[u];
    }
  }
  return zero != 0.f;
}

// The zeros that pad the image, and in the data gradient those between its rows, are multiplied like everything else; that
// is the same sum unless the other factor is an infinity or a NaN.  Forward, such a filter gives NaN at the borders, as a
// zero-padded image does; the data gradient has no padding in its definition, and with such a filter in LDS (`odd`) the
// positions that hold no gradient are left out one by one.

// R: filter height and width; T: output stride; QUADS: see stage_planes (a 1x1 data gradient of stride 2, which has nothing else to do, takes
// 14.3 us without that code in it and 16.4 with it: 53 images, 40 filters of 18 x 14 onto 48 channels, eight groups)
template <class S, int R, int T, int QUADS>
__global__ __launch_bounds__(GT) void k_group_conv(const typename S::elem *__restrict__ src, const typename S::elem *__restrict__ W,
                                                   const typename S::elem *__restrict__ bias, typename S::elem *__restrict__ dst,
                                                   const GroupArgs a) {
  extern __shared__ float lds[];
  __shared__ int odd;
  constexpr int RS = R * R;
  if (a.flip) {
    if (threadIdx.x == 0) odd = 0;
    __syncthreads();
  }
  const int u0 = int(blockIdx.x) * a.UB, p0 = int(blockIdx.y) * a.TP;
  const int ub = a.units - u0 < a.UB ? a.units - u0 : a.UB;
  float *image = lds, *filt = lds + a.UB * a.cs * a.VR * a.VC;
  stage_planes<S, QUADS>(image, a, buffer_of<S>(src, a.src_bytes), u0 * a.cs, a.UB * a.cs, 1, ub * a.cs, p0 * T);
  // filters as [unit][destination channel][source channel][tap]
  const int nf = ub * a.cd * a.cs * RS;
  for (int i = threadIdx.x; i < nf; i += GT) {
    const int q = a.d_taps.div(i), tap = i - q * RS;
    const int q2 = a.d_cs.div(q), cl = q - q2 * a.cs;
    const int ul = a.d_cd.div(q2), m = q2 - ul * a.cd;
    const int unit = u0 + ul, g = unit - a.d_G.div(unit) * a.G;
    const float f = S::ld(W + (a.flip ? (long(g * a.cs + cl) * a.cd + m) * RS + (RS - 1 - tap)
                                      : (long(g * a.cd + m) * a.cs + cl) * RS + tap));
    filt[i] = f;
    if (a.flip && !isfinite(f)) odd = 1;
  }
  __syncthreads();
  const bool select = a.flip && odd != 0;
  const int strips = (a.TP + STRIP - 1) / STRIP;
  const int items = ub * a.cd * strips * a.DW;
  for (int it = threadIdx.x; it < items; it += GT) {
    const int r1 = a.d_dw.div(it), q = it - r1 * a.DW;
    const int r2 = a.d_strips.div(r1), st = r1 - r2 * strips;
    const int ul = a.d_cd.div(r2), m = r2 - ul * a.cd;
    const int unit = u0 + ul;
    float acc[STRIP];
    float b = 0.f;
    if (bias) b = S::ld(bias + (unit - a.d_G.div(unit) * a.G) * a.cd + m);
#pragma unroll
    for (int o = 0; o < STRIP; ++o) acc[o] = 0.f;
    const float *im = image + (ul * a.cs * a.VR + st * STRIP * T) * a.VC + q * T;
    const float *wf = filt + (ul * a.cd + m) * a.cs * RS;
    for (int cl = 0; cl < a.cs; ++cl) {
      float w[RS];
#pragma unroll
      for (int k = 0; k < RS; ++k) w[k] = wf[k];
      if (T > 1 || !select) {   // (T > 1: forward passes only)
#pragma unroll
        for (int i = 0; i < (STRIP - 1) * T + R; ++i) {
#pragma unroll
          for (int s = 0; s < R; ++s) {
            const float v = im[i * a.VC + s];
#pragma unroll
            for (int r = 0; r < R; ++r)
              if (i >= r && (i - r) % T == 0 && (i - r) / T < STRIP) acc[(i - r) / T] = fmaf(w[r * R + s], v, acc[(i - r) / T]);
          }
        }
      } else {   // (in loops: this path is small rather than fast)
        const int y0 = p0 + st * STRIP - a.padh, x0 = q - a.padw;
#pragma unroll
        for (int o = 0; o < STRIP; ++o) {
#pragma unroll 1
          for (int k = 0; k < RS; ++k) {
            const int r = k / R, s = k - r * R, yy = y0 + o + r, xx = x0 + s;
            const int y = a.d_dil.div(yy < 0 ? 0 : yy), x = a.d_dil.div(xx < 0 ? 0 : xx);
            const bool there = yy >= 0 && y < a.SH && y * a.dil == yy && xx >= 0 && x < a.SW && x * a.dil == xx;
            if (there) acc[o] = fmaf(wf[k], im[(o + r) * a.VC + s], acc[o]);
          }
        }
      }
      im += a.VR * a.VC, wf += RS;
    }
    const int p = p0 + st * STRIP;
    const int pe = a.DH < p0 + a.TP ? a.DH : p0 + a.TP;
    typename S::elem *out = dst + (long(unit * a.cd + m) * a.DH + p) * a.DW + q;
#pragma unroll
    for (int o = 0; o < STRIP; ++o)
      if (p + o < pe) S::st(out + o * a.DW, acc[o] + b);
  }
}

// One (filter k, channel c of its group) pair per blockIdx.x, a chunk of the images per blockIdx.y.  `a` describes the
// staging of x (source) against the pixels of dy (destination); a.UB images are staged together, one channel of each.
// The rows of a strip that lie beyond the last row of dy count as zeros of dy; from the first infinity or NaN that the
// workgroup meets in x on (`odd`), their products are left out instead.
template <class S, int R, int T>
__global__ __launch_bounds__(GT) void k_group_wgrad(const typename S::elem *__restrict__ x, const typename S::elem *__restrict__ dy,
                                                    float *__restrict__ part, typename S::elem *__restrict__ dW,
                                                    const GroupArgs a, int N, int images, unsigned dy_bytes) {
  extern __shared__ float lds[];
  constexpr int RS = R * R;
  __shared__ float red[GT / SGH_WAVE][RS];
  __shared__ int odd;
  if (threadIdx.x == 0) odd = 0;
  const int pair = blockIdx.x, k = a.d_cs.div(pair), cl = pair - k * a.cs, g = a.d_cd.div(k);
  const int C = a.G * a.cs, K = a.G * a.cd;
  const int n_end = (int(blockIdx.y) + 1) * images < N ? (int(blockIdx.y) + 1) * images : N;
  const rsrc_t xs = buffer_of<S>(x, a.src_bytes), ys = buffer_of<S>(dy, dy_bytes);
  const int strips = (a.TP + STRIP - 1) / STRIP;
  float acc[RS];
#pragma unroll
  for (int i = 0; i < RS; ++i) acc[i] = 0.f;
  for (int n0 = int(blockIdx.y) * images; n0 < n_end; n0 += a.UB) {
    const int ub = n_end - n0 < a.UB ? n_end - n0 : a.UB;
    for (int p0 = 0; p0 < a.DH; p0 += a.TP) {
      const int items = ub * strips * a.DW, pe = a.DH < p0 + a.TP ? a.DH : p0 + a.TP;
      struct Item {
        float d[STRIP];
        int p, first, image;
      };
      auto request = [&](int it) {
        Item w;
        const int r1 = a.d_dw.div(it), q = it - r1 * a.DW;
        const int ul = a.d_strips.div(r1), st = r1 - ul * strips;
        w.p = p0 + st * STRIP;
        w.first = (((n0 + ul) * K + k) * a.DH + w.p) * a.DW + q;
        w.image = (ul * a.VR + st * STRIP * T) * a.VC + q * T;
#pragma unroll
        for (int o = 0; o < STRIP; ++o) w.d[o] = ld_elem<S>(ys, w.first + o * a.DW, it < items && w.p + o < pe);
        return w;
      };
      // Up to 3x3 dy is requested before x, not behind the barrier, and one item ahead from there on: 12 -> 10.2 us.  With 25 sums and
      // more that costs the registers of one or two wavefronts per SIMD, as do four loads of four columns in flight with 25: 5x5 on
      // 28 x 91 x 25 x 27 17.1 us as here, 22.3 with both.
      constexpr bool AHEAD = R <= 3;
      [[maybe_unused]] Item next;
      if constexpr (AHEAD) next = request(threadIdx.x);
      __syncthreads();   // (the previous tile has been read)
      if (stage_planes<S, R == 5 ? 2 : 4>(lds, a, xs, n0 * C + g * a.cs + cl, a.UB, C, ub, p0 * T)) odd = 1;
      __syncthreads();
      const bool select = odd != 0;
      for (int it = threadIdx.x; it < items; it += GT) {
        Item w;
        if constexpr (AHEAD) w = next, next = request(it + GT);
        else w = request(it);
        const float *im = lds + w.image;
        if (!select) {
#pragma unroll
          for (int i = 0; i < (STRIP - 1) * T + R; ++i) {
#pragma unroll
            for (int s = 0; s < R; ++s) {
              const float v = im[i * a.VC + s];
#pragma unroll
              for (int r = 0; r < R; ++r)
                if (i >= r && (i - r) % T == 0 && (i - r) / T < STRIP) acc[r * R + s] = fmaf(w.d[(i - r) / T], v, acc[r * R + s]);
            }
          }
        } else {
#pragma unroll 1
          for (int o = 0; o < STRIP && w.p + o < pe; ++o) {
            const float dd = ld_elem<S>(ys, w.first + o * a.DW, true);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
              for (int s = 0; s < R; ++s) acc[r * R + s] = fmaf(dd, im[(o * T + r) * a.VC + s], acc[r * R + s]);
          }
        }
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < RS; ++i) {
    const float v = sgh_wave_sum(acc[i]);
    if (lane == 0) red[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < RS) {
    float v = red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < GT / SGH_WAVE; ++w) v += red[w][threadIdx.x];
    const int pairs = gridDim.x;
    if (gridDim.y == 1) S::st(dW + long(pair) * RS + threadIdx.x, v);
    else part[(long(blockIdx.y) * pairs + pair) * RS + threadIdx.x] = v;
  }
}

template <class S>
__global__ __launch_bounds__(64) void k_group_wgrad_reduce(const float *__restrict__ part, typename S::elem *__restrict__ dW, int n,
                                                           int chunks) {
  const int i = int(blockIdx.x) * 64 + int(threadIdx.x);
  if (i >= n) return;
  float v = 0.f;
  constexpr int U = 8;
  int z = 0;
  for (; z + U <= chunks; z += U) {   // (eight loads in flight, added in chunk order)
    float r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = part[long(z + u) * n + i];
#pragma unroll
    for (int u = 0; u < U; ++u) v += r[u];
  }
  for (; z < chunks; ++z) v += part[long(z) * n + i];
  S::st(dW + i, v);
}

inline size_t unit_bytes(const GroupArgs &a, int channels) { return size_t(channels) * a.VR * a.VC * sizeof(float); }

// The tile of `a` (strides, channels and planes set): as many output rows as fit the LDS target (at least one strip), then
// as many units as give two items to every thread, at most `most`.  False when not even one strip fits.
bool plan_tile(GroupArgs *a, int R, int T, int channels, int out_channels, size_t filter_bytes, int most) {
  a->VC = (a->DW - 1) * T + R;
  int strips = (a->DH + STRIP - 1) / STRIP;
  for (;; strips = (strips + 1) / 2) {
    a->VR = (strips * STRIP - 1) * T + R;
    if (unit_bytes(*a, channels) + filter_bytes <= size_t(kLdsTarget) || strips == 1) break;
  }
  if (unit_bytes(*a, channels) + filter_bytes > size_t(kLdsMost)) return false;
  a->TP = strips * STRIP < a->DH ? strips * STRIP : a->DH;
  const int items = out_channels * strips * a->DW;
  long ub = (2 * GT + items - 1) / items;
  const long fit = long(kLdsTarget / (unit_bytes(*a, channels) + filter_bytes));
  if (ub > fit) ub = fit;
  if (ub > most) ub = most;
  a->UB = ub < 1 ? 1 : int(ub);
  const int read = a->SW < a->VC - a->padw ? a->SW : a->VC - a->padw;   // (a strided layer may leave the last columns out)
  a->QN = a->dil == 1 && a->SW >= 4 && read > 0 ? (read + 3) / 4 : 0;
  a->d_qn = sgh_fastdiv(a->QN ? a->QN : 1);
  a->d_vc = sgh_fastdiv(a->VC), a->d_vr = sgh_fastdiv(a->VR), a->d_cs = sgh_fastdiv(a->cs), a->d_dw = sgh_fastdiv(a->DW);
  a->d_strips = sgh_fastdiv(strips), a->d_cd = sgh_fastdiv(a->cd), a->d_dil = sgh_fastdiv(a->dil), a->d_G = sgh_fastdiv(a->G);
  a->d_taps = sgh_fastdiv(R * R);
  return true;
}

struct Plan {
  GroupArgs a;
  int R, T;                 // filter size, output stride of the kernel
  size_t lds;
  int images, chunks;       // weight gradient: images per chunk
};

bool make_plan(const sgh_conv_geom *g, int which, int elem, Plan *p) {
  if (g->groups < 2) return false;
  const int cg = g->C / g->groups, kg = g->K / g->groups;
  if (cg > kNarrow || kg > kNarrow) return false;
  if (g->R != g->S || (g->R != 1 && g->R != 3 && g->R != 5 && g->R != 7)) return false;
  if (g->stride_h != g->stride_w || g->stride_h > 2 || g->pad_h >= g->R || g->pad_w >= g->R) return false;
  GroupArgs &a = p->a;
  a = GroupArgs();
  p->R = g->R;
  const bool dgrad = which == SGH_CONV_DGRAD;
  p->T = dgrad ? 1 : g->stride_h;
  a.G = g->groups, a.units = g->N * g->groups, a.flip = dgrad;
  if (dgrad) {
    a.cs = kg, a.cd = cg, a.SH = g->P, a.SW = g->Q, a.DH = g->H, a.DW = g->W;
    a.dil = g->stride_h, a.padh = g->R - 1 - g->pad_h, a.padw = g->S - 1 - g->pad_w;
  } else {
    a.cs = cg, a.cd = kg, a.SH = g->H, a.SW = g->W, a.DH = g->P, a.DW = g->Q;
    a.dil = 1, a.padh = g->pad_h, a.padw = g->pad_w;
  }
  a.src_bytes = unsigned(size_t(a.units) * a.cs * a.SH * a.SW * elem);
  p->images = g->N, p->chunks = 1;
  if (which == SGH_CONV_WGRAD) {
    if (!plan_tile(&a, p->R, p->T, 1, 1, 0, g->N)) return false;
    p->lds = unit_bytes(a, 1) * a.UB;
    // eight workgroups per CU, every chunk a whole number of stagings
    const long pairs = long(g->K) * cg, want = (8L * sgh_num_cus() + pairs - 1) / pairs;
    const long stagings = (g->N + a.UB - 1) / a.UB;
    const long chunks = want < stagings ? want : stagings;
    p->images = int((stagings + chunks - 1) / chunks) * a.UB;
    p->chunks = (g->N + p->images - 1) / p->images;
    return p->chunks <= 65535;
  }
  const size_t filter = size_t(a.cs) * a.cd * p->R * p->R * sizeof(float);
  if (!plan_tile(&a, p->R, p->T, a.cs, a.cd, filter, a.units)) return false;
  p->lds = (unit_bytes(a, a.cs) + filter) * a.UB;
  return (a.DH + a.TP - 1) / a.TP <= 65535;
}

template <class S, int R, int T>
void launch(const Plan &p, const sgh_conv_geom *g, int which, const void *a, const void *b, const void *bias, void *out, void *ws,
            hipStream_t s) {
  typedef typename S::elem E;
  const E *ea = static_cast<const E *>(a), *eb = static_cast<const E *>(b);
  E *eo = static_cast<E *>(out);
  if (which != SGH_CONV_WGRAD) {
    const dim3 grid((p.a.units + p.a.UB - 1) / p.a.UB, (p.a.DH + p.a.TP - 1) / p.a.TP);
    auto kern = k_group_conv<S, R, T, 4>;
    if constexpr (R == 1)
      if (!p.a.QN) kern = k_group_conv<S, R, T, 0>;
    hipLaunchKernelGGL(kern, grid, dim3(GT), p.lds, s, ea, eb, static_cast<const E *>(bias), eo, p.a);
    return;
  }
  const int pairs = g->K * p.a.cs, n = pairs * R * R;
  float *part = static_cast<float *>(ws);
  const unsigned dy_bytes = unsigned(size_t(g->N) * g->K * g->P * g->Q * sizeof(E));
  hipLaunchKernelGGL((k_group_wgrad<S, R, T>), dim3(pairs, p.chunks), dim3(GT), p.lds, s, eb, ea, part, eo, p.a, g->N, p.images,
                     dy_bytes);
  if (p.chunks > 1)
    hipLaunchKernelGGL(k_group_wgrad_reduce<S>, dim3((n + 63) / 64), dim3(64), 0, s, part, eo, n, p.chunks);
}

template <class S>
void dispatch(const Plan &p, const sgh_conv_geom *g, int which, const void *a, const void *b, const void *bias, void *out, void *ws,
              hipStream_t s) {
#define SGH_GROUP_CASE(R_)                                                                     \
  case R_:                                                                                     \
    if (p.T == 1) launch<S, R_, 1>(p, g, which, a, b, bias, out, ws, s);                       \
    else launch<S, R_, 2>(p, g, which, a, b, bias, out, ws, s);                                \
    break;
  switch (p.R) {
    SGH_GROUP_CASE(1)
    SGH_GROUP_CASE(3)
    SGH_GROUP_CASE(5)
    SGH_GROUP_CASE(7)
  }
#undef SGH_GROUP_CASE
}

}  // namespace

bool sgh_group_conv_supported(const sgh_conv_geom *g, int which) {
  Plan p;
  return make_plan(g, which, 4, &p);
}

size_t sgh_group_conv_workspace_bytes(const sgh_conv_geom *g, int which) {
  Plan p;
  if (which != SGH_CONV_WGRAD || !make_plan(g, which, 4, &p) || p.chunks == 1) return 0;
  return size_t(p.chunks) * g->K * p.a.cs * p.R * p.R * sizeof(float);
}

int sgh_group_conv_run(const sgh_conv_geom *g, int which, int dtype, const void *a, const void *b, const void *bias, void *out,
                       void *workspace, size_t ws_bytes, hipStream_t s) {
  Plan p;
  if (!make_plan(g, which, dtype == 0 ? 4 : 2, &p)) return SGH_EUNSUPPORTED;
  if (p.chunks > 1 && (!workspace || ws_bytes < sgh_group_conv_workspace_bytes(g, which))) return SGH_EWORKSPACE;
  if (dtype == 0) dispatch<StF32>(p, g, which, a, b, bias, out, workspace, s);
  else if (dtype == 1) dispatch<StF16>(p, g, which, a, b, bias, out, workspace, s);
  else dispatch<StBF16>(p, g, which, a, b, bias, out, workspace, s);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}
