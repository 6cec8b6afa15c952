// Pooling forward/backward for NCHW fp32.
//
// Max-pool backward is a gather: one thread owns one dx element, visits the (at most
// ceil(kh/sh) * ceil(kw/sw)) windows that contain it in ascending (p, q) order, recomputes each
// window's first maximum (row-major scan, strict '>') and adds dy when the maximum sits on its
// own element.  The additions therefore happen in exactly the order of the CPU scatter loop, so
// dx is bit-identical to it and no atomics are needed.
#include "common.h"
#include "fastdiv.h"
#include "storage.h"

namespace {

constexpr int kBlock = 256;

struct PoolG {
  int H, W, P, Q, kh, kw, sh, sw, ph, pw;
};

// flat index (h * W + w) of the first maximum of window (p, q) in plane `b`; -1 if empty
template <class S>
__device__ __forceinline__ int window_argmax(const typename S::elem *__restrict__ b, const PoolG g, int p, int q,
                                             float *best_out) {
  int hs = p * g.sh - g.ph, ws = q * g.sw - g.pw;
  const int he = min(hs + g.kh, g.H), we = min(ws + g.kw, g.W);
  hs = max(hs, 0);
  ws = max(ws, 0);
  float best = -3.402823466e38f;
  int bi = -1;
  for (int h = hs; h < he; ++h)
    for (int w = ws; w < we; ++w) {
      const float v = S::ld(b + h * g.W + w);
      if (v > best) {
        best = v;
        bi = h * g.W + w;
      }
    }
  if (best_out) *best_out = best;
  return bi;
}

template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_max_fwd(const typename S::elem *__restrict__ x,
                                                        typename S::elem *__restrict__ y, PoolG g, size_t total) {
  const size_t stride = size_t(gridDim.x) * kBlock;
  const int PQ = g.P * g.Q;
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const size_t plane = i / PQ;
    const int r = int(i - plane * PQ);
    float best;
    window_argmax<S>(x + plane * size_t(g.H) * g.W, g, r / g.Q, r % g.Q, &best);
    S::st(y + i, best);
  }
}

// The residual networks' pooling layer (3 x 3, stride 2, padding 1, even image, Q a multiple of the vector
// length): a thread produces one vector of outputs from two vectors and one element of each of its three input
// rows, comparing in the order of window_argmax (rows top to bottom, columns left to right, strict '>').
template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_max_fwd_3x3s2(const typename S::elem *__restrict__ x,
                                                              typename S::elem *__restrict__ y, int H, int W, size_t nvec) {
  constexpr int V = S::VEC;
  const int P = H >> 1, Q = W >> 1, QV = Q / V;
  const float none = -__builtin_inff();   // (never greater than anything: a position outside the image)
  const size_t stride = size_t(gridDim.x) * kBlock;
  for (size_t iv = size_t(blockIdx.x) * kBlock + threadIdx.x; iv < nvec; iv += stride) {
    const size_t pr = iv / QV;              // plane * P + p
    const int qv = int(iv - pr * QV), q = qv * V;
    const size_t plane = pr / P;
    const int p = int(pr - plane * P);
    const typename S::elem *xb = x + plane * size_t(H) * W;
    float best[V];
#pragma unroll
    for (int j = 0; j < V; ++j) best[j] = -3.402823466e38f;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int h = 2 * p - 1 + r;
      if (h < 0) continue;                  // (h <= H - 1 always: H is even)
      const typename S::elem *row = xb + size_t(h) * W + 2 * q;
      float e[2 * V + 1];
      e[0] = q > 0 ? S::ld(row - 1) : none;
      S::template load16<false>(row, e + 1);
      S::template load16<false>(row + V, e + 1 + V);
#pragma unroll
      for (int j = 0; j < V; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (e[2 * j + c] > best[j]) best[j] = e[2 * j + c];
    }
    S::store16(y + (pr * size_t(Q)) + q, best);
  }
}

template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_max_bwd(const typename S::elem *__restrict__ dy,
                                                        const typename S::elem *__restrict__ x,
                                                        typename S::elem *__restrict__ dx, PoolG g, size_t total) {
  const size_t stride = size_t(gridDim.x) * kBlock;
  const int HW = g.H * g.W, PQ = g.P * g.Q;
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const size_t plane = i / HW;
    const int r = int(i - plane * HW);
    const int h = r / g.W, w = r - h * g.W;
    const typename S::elem *xb = x + plane * size_t(HW);
    const typename S::elem *db = dy + plane * size_t(PQ);
    // windows p with p*sh - ph <= h < p*sh - ph + kh
    const int hp = h + g.ph, wp = w + g.pw;
    const int p_lo = hp < g.kh ? 0 : (hp - g.kh) / g.sh + 1;
    const int p_hi = min(hp / g.sh, g.P - 1);
    const int q_lo = wp < g.kw ? 0 : (wp - g.kw) / g.sw + 1;
    const int q_hi = min(wp / g.sw, g.Q - 1);
    float s = 0.f;
    for (int p = p_lo; p <= p_hi; ++p)
      for (int q = q_lo; q <= q_hi; ++q)
        if (window_argmax<S>(xb, g, p, q, nullptr) == r) s += S::ld(db + p * g.Q + q);
    S::st(dx + i, s);
  }
}

// ---- 3 x 3 windows, stride 2, padding 1 (the residual networks' pooling layer) on planes of any size ------------------
// One lane per window column, everything in registers: a lane loads the pair (2 q, 2 q + 1) of an x row -- four bytes of
// 16-bit elements, eight of fp32, the lanes of a row contiguous, at whatever alignment the row has -- and takes element 2 q - 1
// from the lane before it.  GROUP lanes form a strip of up to kStrip window rows of one plane (8, 16, 32 or 64 by the plane's
// width, so that narrow planes do not leave lanes idle); the loads of a strip are all requested before the first is used.
// Rows or columns outside the image read as -inf, which no comparison selects.  Planes wider than GROUP windows are cut
// into chunks that overlap by one lane on either side.
//
// The kernels that the odd sizes ran before staged elements one by one in LDS (backward) or gave every output its own nine
// loads (forward): bfloat16 50 x 72 x 57 x 43, 40.7 + 18.8 us; here 17.6 + 9.2.  Backward of the residual networks' stem
// (N x 64 x 112 x 112) against rows staged in LDS as whole vectors: bfloat16 N = 64 65.8 -> 53.0, 128 125 -> 107, fp32 N = 64
// 82.3 -> 82.8.
constexpr int kStrip = 7;
constexpr float kLowest = -3.402823466e38f;

struct RowBest {
  float m;
  int k;   // column within the window (0..2), 64 = none
};

__device__ __forceinline__ RowBest best_of(float a, float b, float c) {   // first maximum of a window's row
  RowBest r{kLowest, 64};
  if (a > r.m) r.m = a, r.k = 0;
  if (b > r.m) r.m = b, r.k = 1;
  if (c > r.m) r.m = c, r.k = 2;
  return r;
}

struct StripG {
  int H, W, P, Q;
  int rows;               // window rows per strip
  int strips, chunks;     // per plane
  int units;              // planes * strips * chunks
  unsigned x_bytes, y_bytes;
  sgh_fastdiv d_chunks, d_strips;
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;

// Two neighbouring elements as stored; `ok` false: nothing is read
template <class S>
struct Pair {
  typedef typename S::elem elem;
  float lo, hi;
  static __device__ __forceinline__ Pair load(rsrc_t r, int elem_index, bool ok) {
    const int off = ok ? elem_index * int(sizeof(elem)) : int(0x80000000u);
    if constexpr (sizeof(elem) == 4) {
      typedef unsigned int u2 __attribute__((ext_vector_type(2)));
      const u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
      const unsigned a = v[0], b = v[1];   // (copies: a bit cast of a vector's element takes element 0)
      return Pair{__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)};
    } else {
      const unsigned v = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
      const elem a = elem(v & 0xffffu), b = elem(v >> 16);
      return Pair{S::ld(&a), S::ld(&b)};
    }
  }
};

template <class S>
__device__ __forceinline__ float ld_one(rsrc_t r, int elem_index, bool ok) {
  typedef typename S::elem elem;
  const int off = ok ? elem_index * int(sizeof(elem)) : int(0x80000000u);
  if constexpr (sizeof(elem) == 4) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else {
    const elem e = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
    return S::ld(&e);
  }
}

// What the lanes of a wavefront work on: strip of `rows` window rows from p0 of plane `plane`, window column q
template <int GROUP>
struct Strip {
  int plane, p0, q;
  bool live, inside, makes;   // a strip at all; the window exists; this lane produces its results (not a halo lane)
  __device__ __forceinline__ Strip(const StripG &g) {
    const int lane = threadIdx.x & 63, l = lane & (GROUP - 1);
    const int unit = (int(blockIdx.x) * (kBlock / 64) + int(threadIdx.x >> 6)) * (64 / GROUP) + lane / GROUP;
    live = unit < g.units;
    const int u = live ? unit : 0;
    const int t = g.d_chunks.div(u), chunk = u - t * g.chunks;
    plane = g.d_strips.div(t);
    p0 = (t - plane * g.strips) * g.rows;
    const bool halo = g.chunks > 1;
    q = halo ? chunk * (GROUP - 2) + l - 1 : l;
    inside = live && q >= 0 && q < g.Q;
    makes = inside && (!halo || (l > 0 && l < GROUP - 1));
  }
};

// The three elements of x row h that window column q reads
template <class S, int GROUP>
struct Row3 {
  float a, b, c;
  // requested: the pair (2 q, 2 q + 1), or in a last column of an odd row the pair before it
  static __device__ __forceinline__ Pair<S> request(rsrc_t x, const StripG &g, const Strip<GROUP> &s, int h) {
    const bool ok = s.inside && h >= 0 && h < g.H;
    const int w = 2 * s.q + 1 < g.W ? 2 * s.q : 2 * s.q - 1;
    return Pair<S>::load(x, (s.plane * g.H + h) * g.W + w, ok);
  }
  __device__ __forceinline__ Row3(const Pair<S> &v, const StripG &g, const Strip<GROUP> &s, int h) {
    const float none = -__builtin_inff();
    const bool ok = s.inside && h >= 0 && h < g.H, whole = 2 * s.q + 1 < g.W;
    b = !ok ? none : whole ? v.lo : v.hi;
    c = ok && whole ? v.hi : none;
    const float left = __shfl_up(c, 1, GROUP);
    a = s.q > 0 && (threadIdx.x & (GROUP - 1)) != 0 ? left : none;
    if (!ok) a = none;
  }
};

// a 2 x 2 block of dx, two neighbouring elements per store; `below` / `right`: whether the second row / column exists
template <class S>
__device__ __forceinline__ void store_block(typename S::elem *o, int W, bool below, bool right, float o00, float o01, float o10,
                                            float o11) {
  typedef typename S::elem elem;
  elem e[4];
  S::st(e, o00), S::st(e + 1, o01), S::st(e + 2, o10), S::st(e + 3, o11);
  if (right) {   // (at the alignment of an element)
    if constexpr (sizeof(elem) == 4) {
      typedef float pair __attribute__((ext_vector_type(2), aligned(4)));
      *reinterpret_cast<pair *>(o) = pair{e[0], e[1]};
      if (below) *reinterpret_cast<pair *>(o + W) = pair{e[2], e[3]};
    } else {
      typedef unsigned pair __attribute__((aligned(2)));
      *reinterpret_cast<pair *>(o) = unsigned(e[0]) | (unsigned(e[1]) << 16);
      if (below) *reinterpret_cast<pair *>(o + W) = unsigned(e[2]) | (unsigned(e[3]) << 16);
    }
  } else {
    o[0] = e[0];
    if (below) o[W] = e[2];
  }
}

template <class S, int GROUP>
__global__ __launch_bounds__(kBlock) void k_pool_max_fwd_strip(const typename S::elem *__restrict__ x,
                                                              typename S::elem *__restrict__ y, const StripG g) {
  typedef typename S::elem elem;
  const Strip<GROUP> s(g);
  const rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(x), 0, g.x_bytes, 0x00020000);
  constexpr int NR = 2 * kStrip + 1;
  Pair<S> v[NR];
  const int h0 = 2 * s.p0 - 1;
#pragma unroll
  for (int j = 0; j < NR; ++j) v[j] = Row3<S, GROUP>::request(xr, g, s, j <= 2 * g.rows ? h0 + j : -1);
  elem *out = y + (size_t(s.plane) * g.P + s.p0) * g.Q + s.q;
  const Row3<S, GROUP> r0(v[0], g, s, h0);
  float top = best_of(r0.a, r0.b, r0.c).m;
#pragma unroll
  for (int k = 0; k < kStrip; ++k) {
    if (k >= g.rows) break;
    const Row3<S, GROUP> rm(v[2 * k + 1], g, s, h0 + 2 * k + 1), rb(v[2 * k + 2], g, s, h0 + 2 * k + 2);
    const float mid = best_of(rm.a, rm.b, rm.c).m, bot = best_of(rb.a, rb.b, rb.c).m;
    float best = top;
    if (mid > best) best = mid;
    if (bot > best) best = bot;
    top = bot;
    if (s.makes && s.p0 + k < g.P) S::st(out + size_t(k) * g.Q, best);
  }
}

// The dx block (rows 2 i, 2 i + 1; columns 2 j, 2 j + 1) can only receive from windows (i, j), (i, j + 1), (i + 1, j),
// (i + 1, j + 1), and only at fixed positions of those windows:
//   * window p shares its top row with window p - 1's bottom row: the per-row first maximum (strict '>',
//     left to right) is computed once per x row, and three of them combine top to bottom -- the same winner
//     as the row-major scan of the CPU loop;
//   * the winner is kept as a code 3 * dh + dw; the right-hand neighbour's code and dy come from lane + 1;
//   * a block's four elements add the dy of the windows whose code names them, in ascending (p, q) order
//     starting from +0.0, exactly the additions of the CPU's scatter loop.
// A strip also computes the window row below it.
template <class S, int GROUP>
__global__ __launch_bounds__(kBlock) void k_pool_max_bwd_strip(const typename S::elem *__restrict__ dy,
                                                              const typename S::elem *__restrict__ x,
                                                              typename S::elem *__restrict__ dx, const StripG g) {
  typedef typename S::elem elem;
  const Strip<GROUP> s(g);
  const rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(x), 0, g.x_bytes, 0x00020000);
  const rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(dy), 0, g.y_bytes, 0x00020000);
  constexpr int NR = 2 * kStrip + 3;
  Pair<S> v[NR];
  float d[kStrip + 1];
  const int h0 = 2 * s.p0 - 1;
#pragma unroll
  for (int k = 0; k <= kStrip; ++k)
    d[k] = ld_one<S>(yr, (s.plane * g.P + s.p0 + k) * g.Q + s.q, s.inside && k <= g.rows && s.p0 + k < g.P);
#pragma unroll
  for (int j = 0; j < NR; ++j) v[j] = Row3<S, GROUP>::request(xr, g, s, j <= 2 * g.rows + 2 ? h0 + j : -1);
  const bool last = (threadIdx.x & (GROUP - 1)) == GROUP - 1;   // no lane to the right (a halo lane, or the plane's last window)
  const Row3<S, GROUP> r0(v[0], g, s, h0);
  RowBest top = best_of(r0.a, r0.b, r0.c);
  int code_p = 64, ncode_p = 64;
  float dy_p = 0.f, ndy_p = 0.f;
#pragma unroll
  for (int k = 0; k <= kStrip; ++k) {
    if (k > g.rows) break;
    const Row3<S, GROUP> rm(v[2 * k + 1], g, s, h0 + 2 * k + 1), rb(v[2 * k + 2], g, s, h0 + 2 * k + 2);
    const RowBest mid = best_of(rm.a, rm.b, rm.c), bot = best_of(rb.a, rb.b, rb.c);
    float best = top.m;
    int code = top.k;
    if (mid.m > best) best = mid.m, code = 3 + mid.k;
    if (bot.m > best) code = 6 + bot.k;
    if (!s.inside || s.p0 + k >= g.P) code = 64;
    top = bot;
    const float dyv = d[k];
    int ncode = __shfl_down(code, 1, GROUP);
    const float ndy = __shfl_down(dyv, 1, GROUP);
    if (last) ncode = 64;
    if (k > 0 && s.makes && s.p0 + k - 1 < g.P) {
      // block row p0 + k - 1: windows (.., q), (.., q + 1), then the two below, in that order
      const float o00 = 0.f + (code_p == 4 ? dy_p : 0.f);
      const float o01 = (0.f + (code_p == 5 ? dy_p : 0.f)) + (ncode_p == 3 ? ndy_p : 0.f);
      const float o10 = (0.f + (code_p == 7 ? dy_p : 0.f)) + (code == 1 ? dyv : 0.f);
      const float o11 = (((0.f + (code_p == 8 ? dy_p : 0.f)) + (ncode_p == 6 ? ndy_p : 0.f)) + (code == 2 ? dyv : 0.f)) +
                        (ncode == 0 ? ndy : 0.f);
      const int h = 2 * (s.p0 + k - 1);
      store_block<S>(dx + (size_t(s.plane) * g.H + h) * g.W + 2 * s.q, g.W, h + 1 < g.H, 2 * s.q + 1 < g.W, o00, o01, o10, o11);
    }
    code_p = code, ncode_p = ncode, dy_p = dyv, ndy_p = ndy;
  }
}

// ---- 2 x 2 windows, stride 2, no padding: the windows do not overlap, so both passes stream -----------------------------
// One thread per 2 x 2 block of x: two pairs in; the maximum (or mean) out, or in the backward pass dy to the element of the
// first maximum (a quarter of dy to each).  Blocks of a last odd row or column belong to no window and receive zero.
// fp32 128 x 32 x 32 x 32, maximum: backward 19.4 -> 6.5 us (was: rows staged in LDS, a table of arg-max positions), forward
// 6.9 -> 4.3 (one thread per output, four loads each); mean of 50 x 72 x 57 x 43 37.4 + 11.8 -> 9.7 + 7.1.
struct QuadG {
  int H, W, P, Q;
  int BW;                 // blocks per row: ceil(W / 2) backward, Q forward
  int total;              // blocks
  unsigned x_bytes;
  sgh_fastdiv d_bw, d_bh;
};

// kQuadReluMax: x is the input of a ReLU in front of the pooling layer; the ReLU is applied as x is read, and its gate as the gradient
// is stored: the bits of the two layers one after the other, without the rectified tensor and its gradient (fp32 128 x 32 x 32 x 32, forward
// and backward: 5.5 + 4.7 + 6.7 + 7.2 us of kernels, 4.5 + 7 here).
enum { kQuadMean, kQuadMax, kQuadReluMax };

template <class S>
__device__ __forceinline__ void rectify(Pair<S> &t, Pair<S> &b) {
  t.lo = t.lo >= 0.f ? t.lo : 0.f, t.hi = t.hi >= 0.f ? t.hi : 0.f;
  b.lo = b.lo >= 0.f ? b.lo : 0.f, b.hi = b.hi >= 0.f ? b.hi : 0.f;
}

template <class S, int MODE>
__global__ __launch_bounds__(kBlock) void k_pool_quad_fwd(const typename S::elem *__restrict__ x, typename S::elem *__restrict__ y,
                                                         const QuadG g) {
  typedef typename S::elem elem;
  constexpr bool MAX = MODE != kQuadMean;
  const rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(x), 0, g.x_bytes, 0x00020000);
  constexpr int U = 4;
  for (int i0 = int(blockIdx.x) * kBlock * U + int(threadIdx.x); i0 < g.total; i0 += int(gridDim.x) * kBlock * U) {
    Pair<S> t[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kBlock, r = g.d_bw.div(i), q = i - r * g.BW, plane = g.d_bh.div(r), p = r - plane * g.P;
      const int at = (plane * g.H + 2 * p) * g.W + 2 * q;
      t[u] = Pair<S>::load(xr, at, i < g.total);
      b[u] = Pair<S>::load(xr, at + g.W, i < g.total);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kBlock;
      if (i >= g.total) break;
      float v;
      if (MAX) {
        v = kLowest;
        if constexpr (MODE == kQuadReluMax) rectify<S>(t[u], b[u]);
        if (t[u].lo > v) v = t[u].lo;
        if (t[u].hi > v) v = t[u].hi;
        if (b[u].lo > v) v = b[u].lo;
        if (b[u].hi > v) v = b[u].hi;
      } else {
        v = ((((0.f + t[u].lo) + t[u].hi) + b[u].lo) + b[u].hi) / 4.f;
      }
      S::st(y + i, v);
    }
  }
}

template <class S, int MODE>
__global__ __launch_bounds__(kBlock) void k_pool_quad_bwd(const typename S::elem *__restrict__ dy, const typename S::elem *__restrict__ x,
                                                         typename S::elem *__restrict__ dx, const QuadG g, int BH, unsigned y_bytes) {
  typedef typename S::elem elem;
  constexpr bool MAX = MODE != kQuadMean;
  const rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(x), 0, MAX ? g.x_bytes : 0, 0x00020000);
  const rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(dy), 0, y_bytes, 0x00020000);
  constexpr int U = 4;
  for (int i0 = int(blockIdx.x) * kBlock * U + int(threadIdx.x); i0 < g.total; i0 += int(gridDim.x) * kBlock * U) {
    Pair<S> t[U], b[U];
    float d[U];
    int at[U], hr[U], q[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * kBlock, r = g.d_bw.div(i), plane = g.d_bh.div(r), p = r - plane * BH;
      q[u] = i - r * g.BW;
      hr[u] = 2 * p;
      at[u] = (plane * g.H + 2 * p) * g.W + 2 * q[u];
      const bool window = i < g.total && p < g.P && q[u] < g.Q;
      d[u] = ld_one<S>(yr, (plane * g.P + p) * g.Q + q[u], window);
      if (MAX) {
        t[u] = Pair<S>::load(xr, at[u], window);
        b[u] = Pair<S>::load(xr, at[u] + g.W, window);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i0 + u * kBlock >= g.total) break;
      float o[4];
      if (MAX) {
        float v = kLowest;
        int k = -1;
        bool open[4] = {true, true, true, true};
        if constexpr (MODE == kQuadReluMax) {
          open[0] = t[u].lo > 0.f, open[1] = t[u].hi > 0.f, open[2] = b[u].lo > 0.f, open[3] = b[u].hi > 0.f;
          rectify<S>(t[u], b[u]);
        }
        if (t[u].lo > v) v = t[u].lo, k = 0;
        if (t[u].hi > v) v = t[u].hi, k = 1;
        if (b[u].lo > v) v = b[u].lo, k = 2;
        if (b[u].hi > v) k = 3;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = open[e] ? 0.f + (k == e ? d[u] : 0.f) : 0.f;   // (a block without a window read d = 0)
      } else {
        o[0] = o[1] = o[2] = o[3] = 0.f + d[u] / 4.f;
      }
      store_block<S>(dx + at[u], g.W, hr[u] + 1 < g.H, 2 * q[u] + 1 < g.W, o[0], o[1], o[2], o[3]);
    }
  }
}

// Tiled max-pool backward: one workgroup owns a band of TH rows of one (n, c) plane of dx.
//   1. the x rows every window touching the band needs and the dy rows of those windows are
//      staged in LDS (both are contiguous runs of the plane: 128-bit copies when aligned),
//   2. each of those windows gets its first-maximum position (flat h * W + w) into LDS,
//   3. each dx element of the band adds dy over the windows that contain it, in ascending (p, q)
//      order, when the window's maximum sits on it -- the same order as the CPU scatter loop.
// The 256 threads form 64 columns x 4 rows, so no per-element division is needed: a thread's
// column window range is fixed, and the per-row window range is computed once per band row.
// x, dy and dx each cross HBM once (plus the band halo of x).
// KH/KW/SH/SW > 0 fix the window at compile time: the scans are then fully unrolled, every LDS
// read of a window or of a dx element is issued before the first compare, and out-of-range
// positions are predicated instead of branched over.  0 = read the geometry at run time.
template <int KH, int KW, int SH, int SW, class S>
__global__ __launch_bounds__(kBlock) void k_pool_max_bwd_tiled(const typename S::elem *__restrict__ dy,
                                                              const typename S::elem *__restrict__ x,
                                                              typename S::elem *__restrict__ dx, PoolG g, int TH,
                                                              int bands, int max_xrows, int max_np) {
  if (KH > 0) {
    g.kh = KH;
    g.kw = KW;
    g.sh = SH;
    g.sw = SW;
  }
  extern __shared__ float smem[];
  float *xs = smem;                                               // [max_xrows][W]
  float *ds = xs + max_xrows * g.W;                               // [max_np][Q]
  int *widx = reinterpret_cast<int *>(ds + max_np * g.Q);         // [max_np][Q]
  int *prange = widx + max_np * g.Q;                              // [TH][2]: first / last window row of a band row
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int plane = blockIdx.x / bands, band = blockIdx.x - plane * bands;
  const int h0 = band * TH, h1 = min(h0 + TH, g.H);
  // windows p with [p*sh - ph, p*sh - ph + kh) overlapping [h0, h1)
  const int lo_num = h0 + g.ph - g.kh + 1;
  const int p_lo = lo_num <= 0 ? 0 : (lo_num + g.sh - 1) / g.sh;
  const int p_hi = min((h1 - 1 + g.ph) / g.sh, g.P - 1);
  const int np = p_hi - p_lo + 1;
  const int xr0 = max(p_lo * g.sh - g.ph, 0), xr1 = min(p_hi * g.sh - g.ph + g.kh, g.H);  // x rows [xr0, xr1)
  const typename S::elem *xb = x + size_t(plane) * g.H * g.W + xr0 * g.W;
  const typename S::elem *db = dy + size_t(plane) * g.P * g.Q + p_lo * g.Q;
  typename S::elem *ob = dx + size_t(plane) * g.H * g.W;
  const int nx = (xr1 - xr0) * g.W, nd = np > 0 ? np * g.Q : 0;
  // 16 bytes of the storage type per access when the run is aligned (LDS holds floats)
  constexpr int V = S::VEC;
  if ((reinterpret_cast<uintptr_t>(xb) & 15u) == 0 && nx % V == 0) {
#pragma unroll 4
    for (int i = threadIdx.x; i < nx / V; i += kBlock) {
      float v[V];
      S::template load16<false>(xb + i * V, v);
#pragma unroll
      for (int j = 0; j < V; ++j) xs[i * V + j] = v[j];
    }
  } else {
    for (int i = threadIdx.x; i < nx; i += kBlock) xs[i] = S::ld(xb + i);
  }
  for (int i = threadIdx.x; i < nd; i += kBlock) ds[i] = S::ld(db + i);
  for (int i = threadIdx.x; i < h1 - h0; i += kBlock) {
    const int hp = h0 + i + g.ph;
    prange[2 * i] = (hp < g.kh ? 0 : (hp - g.kh) / g.sh + 1) - p_lo;
    prange[2 * i + 1] = min(hp / g.sh, g.P - 1) - p_lo;
  }
  __syncthreads();
  for (int pp = ty; pp < np; pp += 4) {
    const int hs0 = (p_lo + pp) * g.sh - g.ph;
    for (int q = tx; q < g.Q; q += 64) {
      const int ws0 = q * g.sw - g.pw;
      float best = -3.402823466e38f;
      int bi = -1;
      if (KH > 0) {
        float v[KH > 0 ? KH * KW : 1];
#pragma unroll
        for (int dh = 0; dh < KH; ++dh)
#pragma unroll
          for (int dw = 0; dw < KW; ++dw) {
            const int h = hs0 + dh, w = ws0 + dw;
            const bool ok = unsigned(h) < unsigned(g.H) && unsigned(w) < unsigned(g.W);
            const float xv = xs[ok ? (h - xr0) * g.W + w : 0];
            v[dh * KW + dw] = ok ? xv : -3.402823466e38f;
          }
#pragma unroll
        for (int dh = 0; dh < KH; ++dh)
#pragma unroll
          for (int dw = 0; dw < KW; ++dw)
            if (v[dh * KW + dw] > best) {
              best = v[dh * KW + dw];
              bi = (hs0 + dh) * g.W + ws0 + dw;
            }
      } else {
        const int hs = max(hs0, 0), he = min(hs0 + g.kh, g.H);
        const int ws = max(ws0, 0), we = min(ws0 + g.kw, g.W);
        for (int h = hs; h < he; ++h)
          for (int w = ws; w < we; ++w) {
            const float v = xs[(h - xr0) * g.W + w];
            if (v > best) {
              best = v;
              bi = h * g.W + w;
            }
          }
      }
      widx[pp * g.Q + q] = bi;
    }
  }
  __syncthreads();
  if (KH > 0) {
    // A thread owns an SH x SW block of dx.  The windows that can contain any of its elements are
    // NBH x NBW consecutive ones; their arg-max positions and dy values are read once and serve
    // the whole block (a window whose maximum sits on element r necessarily contains r, so
    // testing the position is enough).
    constexpr int SHc = KH > 0 ? SH : 1, SWc = KW > 0 ? SW : 1;
    constexpr int NBH = KH > 0 ? (KH + SH - 2) / SHc + 1 : 1, NBW = KW > 0 ? (KW + SW - 2) / SWc + 1 : 1;
    const int nbh = (h1 - h0 + SHc - 1) / SHc, nbw = (g.W + SWc - 1) / SWc;
    for (int bj = tx; bj < nbw; bj += 64) {
      const int w0 = bj * SWc, wp0 = w0 + g.pw;
      const int ql0 = wp0 < g.kw ? 0 : (wp0 - g.kw) / g.sw + 1;
      for (int bi = ty; bi < nbh; bi += 4) {
        const int hb = h0 + bi * SHc, hp0 = hb + g.ph;
        const int pl0 = (hp0 < g.kh ? 0 : (hp0 - g.kh) / g.sh + 1) - p_lo;
        int wi[NBH * NBW];
        float dv[NBH * NBW];
#pragma unroll
        for (int dp = 0; dp < NBH; ++dp)
#pragma unroll
          for (int dq = 0; dq < NBW; ++dq) {
            const bool ok = pl0 + dp < np && ql0 + dq < g.Q;
            const int o = ok ? (pl0 + dp) * g.Q + ql0 + dq : 0;
            wi[dp * NBW + dq] = ok ? widx[o] : -2;
            dv[dp * NBW + dq] = ds[o];
          }
#pragma unroll
        for (int a = 0; a < SHc; ++a) {
          const int h = hb + a;
          if (h >= h1) break;
          float out[SWc];
#pragma unroll
          for (int b2 = 0; b2 < SWc; ++b2) {
            const int r = h * g.W + w0 + b2;
            // s is never -0.0 (it starts at +0.0), so adding +0.0 for a window that does not match
            // leaves it bit-identical to skipping the addition; ascending (p, q) order as on the CPU
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < NBH * NBW; ++i) s += wi[i] == r ? dv[i] : 0.f;
            out[b2] = s;
          }
          typename S::elem *o = ob + h * g.W + w0;
          if (V == 4 && SWc == 2 && w0 + 1 < g.W && (reinterpret_cast<uintptr_t>(o) & 7u) == 0) {
            typedef float v2f __attribute__((ext_vector_type(2)));
            *reinterpret_cast<v2f *>(o) = v2f{out[0], out[SWc - 1]};
          } else {
#pragma unroll
            for (int b2 = 0; b2 < SWc; ++b2)
              if (w0 + b2 < g.W) S::st(o + b2, out[b2]);
          }
        }
      }
    }
  } else {
    for (int w = tx; w < g.W; w += 64) {
      const int wp = w + g.pw;
      const int ql = wp < g.kw ? 0 : (wp - g.kw) / g.sw + 1;
      const int qh = min(wp / g.sw, g.Q - 1);
      for (int hh = ty; hh < h1 - h0; hh += 4) {
        const int r = (h0 + hh) * g.W + w;
        const int pl = prange[2 * hh], ph_ = prange[2 * hh + 1];
        float s = 0.f;
        for (int p = pl; p <= ph_; ++p)
          for (int q = ql; q <= qh; ++q)
            if (widx[p * g.Q + q] == r) s += ds[p * g.Q + q];
        S::st(ob + r, s);
      }
    }
  }
}

__device__ __forceinline__ int window_count(const PoolG g, int p, int q, int *hs_, int *he_, int *ws_, int *we_) {
  int hs = p * g.sh - g.ph, ws = q * g.sw - g.pw;
  const int he = min(hs + g.kh, g.H), we = min(ws + g.kw, g.W);
  hs = max(hs, 0);
  ws = max(ws, 0);
  *hs_ = hs;
  *he_ = he;
  *ws_ = ws;
  *we_ = we;
  return (he - hs) * (we - ws);  // count-exclude-padding
}

template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_avg_fwd(const typename S::elem *__restrict__ x,
                                                        typename S::elem *__restrict__ y, PoolG g, size_t total) {
  const size_t stride = size_t(gridDim.x) * kBlock;
  const int PQ = g.P * g.Q;
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const size_t plane = i / PQ;
    const int r = int(i - plane * PQ);
    const typename S::elem *b = x + plane * size_t(g.H) * g.W;
    int hs, he, ws, we;
    const int cnt = window_count(g, r / g.Q, r % g.Q, &hs, &he, &ws, &we);
    float s = 0.f;
    for (int h = hs; h < he; ++h)
      for (int w = ws; w < we; ++w) s += S::ld(b + h * g.W + w);
    S::st(y + i, s / float(cnt));
  }
}

// One window that is the whole plane, planes of at most 64 elements (global average pooling, 7 x 7): a workgroup
// stages its 256 consecutive planes -- one contiguous run of memory -- in LDS with whole-vector loads and a thread
// sums one plane in the order of the loop above.
template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_avg_fwd_global(const typename S::elem *__restrict__ x,
                                                               typename S::elem *__restrict__ y, int HW, size_t planes) {
  constexpr int V = S::VEC;
  extern __shared__ float xs_f[];   // kBlock * HW
  const size_t plane0 = size_t(blockIdx.x) * kBlock;
  const int np = int(planes - plane0 < size_t(kBlock) ? planes - plane0 : size_t(kBlock)), n = np * HW, t = threadIdx.x;
  const typename S::elem *base = x + plane0 * size_t(HW);
  const int nvec = n / V;
  for (int v = t; v < nvec; v += kBlock) {
    float e[V];
    S::template load16<false>(base + v * V, e);
#pragma unroll
    for (int q = 0; q < V; ++q) xs_f[v * V + q] = e[q];
  }
  for (int i = nvec * V + t; i < n; i += kBlock) xs_f[i] = S::ld(base + i);
  __syncthreads();
  if (t < np) {
    float s = 0.f;
    for (int j = 0; j < HW; ++j) s += xs_f[t * HW + j];
    S::st(y + plane0 + t, s / float(HW));
  }
}

template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_avg_bwd(const typename S::elem *__restrict__ dy,
                                                        typename S::elem *__restrict__ dx, PoolG g, size_t total) {
  const size_t stride = size_t(gridDim.x) * kBlock;
  const int HW = g.H * g.W, PQ = g.P * g.Q;
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const size_t plane = i / HW;
    const int r = int(i - plane * HW);
    const int h = r / g.W, w = r - h * g.W;
    const typename S::elem *db = dy + plane * size_t(PQ);
    const int hp = h + g.ph, wp = w + g.pw;
    const int p_lo = hp < g.kh ? 0 : (hp - g.kh) / g.sh + 1;
    const int p_hi = min(hp / g.sh, g.P - 1);
    const int q_lo = wp < g.kw ? 0 : (wp - g.kw) / g.sw + 1;
    const int q_hi = min(wp / g.sw, g.Q - 1);
    float s = 0.f;
    for (int p = p_lo; p <= p_hi; ++p)
      for (int q = q_lo; q <= q_hi; ++q) {
        int hs, he, ws, we;
        const int cnt = window_count(g, p, q, &hs, &he, &ws, &we);
        s += S::ld(db + p * g.Q + q) / float(cnt);
      }
    S::st(dx + i, s);
  }
}

// One window that is the whole plane (global average pooling): every element of a plane receives
// dy[plane] / (H * W), the same arithmetic as the kernel above, written in whole vectors.
template <class S>
__global__ __launch_bounds__(kBlock) void k_pool_avg_bwd_global(const typename S::elem *__restrict__ dy,
                                                               typename S::elem *__restrict__ dx, int HW, size_t total) {
  constexpr int V = S::VEC;
  const size_t stride = size_t(gridDim.x) * kBlock, tid = size_t(blockIdx.x) * kBlock + threadIdx.x;
  const size_t nvec = total / V;
  const float cnt = float(HW);
  for (size_t iv = tid; iv < nvec; iv += stride) {
    const size_t i0 = iv * V;
    size_t plane = i0 / size_t(HW);
    int r = int(i0 - plane * size_t(HW));
    float gv = 0.f + S::ld(dy + plane) / cnt;
    float o[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      if (r == HW) {
        r = 0;
        ++plane;
        gv = 0.f + S::ld(dy + plane) / cnt;
      }
      o[q] = gv;
      ++r;
    }
    S::store16(dx + i0, o);
  }
  for (size_t i = nvec * V + tid; i < total; i += stride) S::st(dx + i, 0.f + S::ld(dy + i / size_t(HW)) / cnt);
}

inline int grid_for(size_t n) {
  size_t blocks = (n + kBlock - 1) / kBlock;
  const size_t cap = size_t(sgh_num_cus()) * 32;
  if (blocks > cap) blocks = cap;
  return int(blocks < 1 ? 1 : blocks);
}

inline PoolG to_g(const sgh_pool_geom *g) {
  return PoolG{g->H, g->W, g->P, g->Q, g->kernel_h, g->kernel_w, g->stride_h, g->stride_w, g->pad_h, g->pad_w};
}

inline bool geom_ok(const sgh_pool_geom *g) {
  return g && g->N > 0 && g->C > 0 && g->H > 0 && g->W > 0 && g->kernel_h > 0 && g->kernel_w > 0 && g->stride_h > 0 &&
         g->stride_w > 0 && g->pad_h >= 0 && g->pad_w >= 0 && g->P > 0 && g->Q > 0 &&
         g->P == (g->H + 2 * g->pad_h - g->kernel_h) / g->stride_h + 1 &&
         g->Q == (g->W + 2 * g->pad_w - g->kernel_w) / g->stride_w + 1 &&
         // every window must overlap the image, else a max window would be empty
         g->pad_h < g->kernel_h && g->pad_w < g->kernel_w &&
         size_t(g->H) * g->W < 0x7fffffffu;
}

// lanes per strip: the narrowest group that holds a row of windows
inline int strip_group(int Q) { return Q <= 8 ? 8 : Q <= 16 ? 16 : Q <= 32 ? 32 : 64; }

inline bool strip_plan(const sgh_pool_geom *g, int esize, StripG *s) {
  if (g->kernel_h != 3 || g->kernel_w != 3 || g->stride_h != 2 || g->stride_w != 2 || g->pad_h != 1 || g->pad_w != 1 || g->W < 2)
    return false;
  const size_t x = size_t(g->N) * g->C * g->H * g->W * esize;
  if (x >= (size_t(1) << 31)) return false;   // (32-bit byte offsets)
  const int group = strip_group(g->Q);
  s->H = g->H, s->W = g->W, s->P = g->P, s->Q = g->Q;
  s->chunks = g->Q <= group ? 1 : (g->Q + group - 3) / (group - 2);
  // rows: the more, the fewer are computed twice; but a strip is one chain of shuffles, so no more than leave every CU two
  // wavefronts.  Backward against the kernels before, 500 shapes: with strips of seven throughout 1.20 times as fast below
  // 100 000 elements and 1.47 below a million, 19 of 262 slower, down to 0.75 (4.0 -> 5.0 us); with this rule 1.44 and 1.70,
  // two slower.  With one or four wavefronts per CU 1.42 / 1.57 and 1.34 / 1.71.
  const long fill = long(g->N) * g->C * s->chunks * g->P * group / 64 / (2 * sgh_num_cus());
  const int most = fill < 1 ? 1 : fill > kStrip ? kStrip : int(fill);
  s->strips = (g->P + most - 1) / most;
  s->rows = (g->P + s->strips - 1) / s->strips;
  s->units = int(size_t(g->N) * g->C * s->strips * s->chunks);   // (fewer than dx elements)
  s->x_bytes = unsigned(x);
  s->y_bytes = unsigned(size_t(g->N) * g->C * g->P * g->Q * esize);
  s->d_chunks = sgh_fastdiv(s->chunks), s->d_strips = sgh_fastdiv(s->strips);
  return true;
}

inline unsigned strip_blocks(const StripG &s) {
  const int per = kBlock / strip_group(s.Q);
  return unsigned((s.units + per - 1) / per);
}

inline bool quad_plan(const sgh_pool_geom *g, int esize, bool bwd, QuadG *s) {
  if (g->kernel_h != 2 || g->kernel_w != 2 || g->stride_h != 2 || g->stride_w != 2 || g->pad_h != 0 || g->pad_w != 0) return false;
  const size_t x = size_t(g->N) * g->C * g->H * g->W * esize;
  if (x >= (size_t(1) << 31)) return false;
  s->H = g->H, s->W = g->W, s->P = g->P, s->Q = g->Q;
  s->BW = bwd ? (g->W + 1) / 2 : g->Q;
  const int bh = bwd ? (g->H + 1) / 2 : g->P;
  s->total = int(size_t(g->N) * g->C * bh * s->BW);
  s->x_bytes = unsigned(x);
  s->d_bw = sgh_fastdiv(s->BW), s->d_bh = sgh_fastdiv(bh);
  return true;
}

// Tensors of 2 GiB and more, where the kernels with 32-bit offsets apply otherwise: by groups of images
inline int images_per_call(const sgh_pool_geom *g, int esize) {
  const bool strip = g->is_max && g->kernel_h == 3 && g->kernel_w == 3 && g->pad_h == 1 && g->pad_w == 1;
  const bool quad = g->kernel_h == 2 && g->kernel_w == 2 && g->pad_h == 0 && g->pad_w == 0;
  const size_t image = size_t(g->C) * g->H * g->W * esize, most = (size_t(1) << 31) - 1;
  if (!(strip || quad) || g->stride_h != 2 || g->stride_w != 2 || image > most || image * g->N <= most) return g->N;
  return int(most / image);
}

// fp32 forward: outputs from which the strip kernel is the faster one (with 64 planes per image, 13 x 80 x 80 5.6 us before
// and 7.0 with it, 21 x 96 x 96 12.5 and 11.9, 64 x 112 x 112 39.2 and 37.6, 128 x 112 x 112 105 and 93).  In 16 bits the
// whole vectors of k_pool_max_fwd_3x3s2 win throughout: 7.0 us against 11.1, 26.9 against 26.5, 49 against 54.
constexpr size_t kStripFwdMin = size_t(2) << 20;

template <class S>
int pool_fwd(const sgh_pool_geom *g, const typename S::elem *x, typename S::elem *y, void *stream) {
  if (!geom_ok(g) || !x || !y) return SGH_EINVAL;
  const int esize = int(sizeof(typename S::elem)), images = images_per_call(g, esize);
  if (images < g->N) {
    sgh_pool_geom part = *g;
    for (int n = 0; n < g->N; n += images) {
      part.N = g->N - n < images ? g->N - n : images;
      const int rc = pool_fwd<S>(&part, x + size_t(n) * g->C * g->H * g->W, y + size_t(n) * g->C * g->P * g->Q, stream);
      if (rc != SGH_OK) return rc;
    }
    return SGH_OK;
  }
  const size_t total = size_t(g->N) * g->C * g->P * g->Q;
  StripG sg;
  QuadG qg;
  if (g->is_max && g->kernel_h == 3 && g->kernel_w == 3 && g->stride_h == 2 && g->stride_w == 2 && g->pad_h == 1 &&
      g->pad_w == 1 && g->H % 2 == 0 && g->W % 2 == 0 && g->Q % S::VEC == 0 && sgh_aligned16(x) && sgh_aligned16(y) &&
      (esize == 2 || total <= kStripFwdMin))
    hipLaunchKernelGGL(k_pool_max_fwd_3x3s2<S>, dim3(grid_for(total / S::VEC)), dim3(kBlock), 0, sgh_stream_of(stream), x, y,
                       g->H, g->W, total / S::VEC);
  else if (g->is_max && strip_plan(g, esize, &sg)) {
    const int group = strip_group(g->Q);
    auto kern = group == 8    ? k_pool_max_fwd_strip<S, 8>
                : group == 16 ? k_pool_max_fwd_strip<S, 16>
                : group == 32 ? k_pool_max_fwd_strip<S, 32>
                              : k_pool_max_fwd_strip<S, 64>;
    hipLaunchKernelGGL(kern, dim3(strip_blocks(sg)), dim3(kBlock), 0, sgh_stream_of(stream), x, y, sg);
  } else if (quad_plan(g, esize, false, &qg)) {
    auto kern = g->is_max ? k_pool_quad_fwd<S, kQuadMax> : k_pool_quad_fwd<S, kQuadMean>;
    hipLaunchKernelGGL(kern, dim3(grid_for((size_t(qg.total) + 3) / 4)), dim3(kBlock), 0, sgh_stream_of(stream), x, y, qg);
  } else if (g->is_max)
    hipLaunchKernelGGL(k_pool_max_fwd<S>, dim3(grid_for(total)), dim3(kBlock), 0, sgh_stream_of(stream), x, y, to_g(g),
                       total);
  else if (g->P == 1 && g->Q == 1 && g->pad_h == 0 && g->pad_w == 0 && g->kernel_h >= g->H && g->kernel_w >= g->W &&
           g->H * g->W <= 64 && sgh_aligned16(x) && (total + kBlock - 1) / kBlock < 0x7fffffffu)
    hipLaunchKernelGGL(k_pool_avg_fwd_global<S>, dim3(unsigned((total + kBlock - 1) / kBlock)), dim3(kBlock),
                       size_t(kBlock) * g->H * g->W * sizeof(float), sgh_stream_of(stream), x, y, g->H * g->W, total);
  else
    hipLaunchKernelGGL(k_pool_avg_fwd<S>, dim3(grid_for(total)), dim3(kBlock), 0, sgh_stream_of(stream), x, y, to_g(g),
                       total);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}

template <class S>
int pool_bwd(const sgh_pool_geom *g, const typename S::elem *dy, const typename S::elem *x, const typename S::elem *y,
             typename S::elem *dx, void *stream) {
  (void)y;
  if (!geom_ok(g) || !dy || !dx) return SGH_EINVAL;
  if (g->is_max && !x) return SGH_EINVAL;
  const int esize = int(sizeof(typename S::elem)), images = images_per_call(g, esize);
  if (images < g->N) {
    sgh_pool_geom part = *g;
    for (int n = 0; n < g->N; n += images) {
      part.N = g->N - n < images ? g->N - n : images;
      const size_t at = size_t(n) * g->C * g->H * g->W;
      const int rc = pool_bwd<S>(&part, dy + size_t(n) * g->C * g->P * g->Q, x ? x + at : x, y, dx + at, stream);
      if (rc != SGH_OK) return rc;
    }
    return SGH_OK;
  }
  const size_t total = size_t(g->N) * g->C * g->H * g->W;
  // algorithmic bytes: dy and (max pooling) x in, dx out
  sgh_prof_kernel_scope prof(g->is_max ? "pool_bwd/k_pool_max_bwd" : "pool_bwd/k_pool_avg_bwd",
                      double(sizeof(typename S::elem)) *
                          (double(total) * (g->is_max ? 2 : 1) + double(g->N) * g->C * g->P * g->Q),
                      sgh_stream_of(stream));
  StripG sg;
  QuadG qg;
  if (g->is_max && strip_plan(g, esize, &sg)) {
    const int group = strip_group(g->Q);
    auto kern = group == 8    ? k_pool_max_bwd_strip<S, 8>
                : group == 16 ? k_pool_max_bwd_strip<S, 16>
                : group == 32 ? k_pool_max_bwd_strip<S, 32>
                              : k_pool_max_bwd_strip<S, 64>;
    SGH_LAUNCH_TIMED(kern, dim3(strip_blocks(sg)), dim3(kBlock), 0, sgh_stream_of(stream), dy, x, dx, sg);
  } else if (quad_plan(g, esize, true, &qg)) {
    auto kern = g->is_max ? k_pool_quad_bwd<S, kQuadMax> : k_pool_quad_bwd<S, kQuadMean>;
    SGH_LAUNCH_TIMED(kern, dim3(grid_for((size_t(qg.total) + 3) / 4)), dim3(kBlock), 0, sgh_stream_of(stream), dy, x, dx, qg,
                     (g->H + 1) / 2, unsigned(size_t(g->N) * g->C * g->P * g->Q * esize));
  } else if (g->is_max) {
    // band height: about 12 KB of x rows per workgroup (measured optimum: enough workgroups per CU to
    // overlap one's staging with another's scans), bands of equal height
    int TH = 3072 / g->W - g->kernel_h;
    if (TH < 1) TH = 1;
    if (TH > g->H) TH = g->H;
    int bands = (g->H + TH - 1) / TH;
    TH = (g->H + bands - 1) / bands;
    bands = (g->H + TH - 1) / TH;
    const int max_np = (TH + g->kernel_h - 2) / g->stride_h + 2;
    const int max_xrows = (max_np - 1) * g->stride_h + g->kernel_h;
    const size_t lds = (size_t(max_xrows) * g->W + size_t(2) * max_np * g->Q + size_t(2) * TH) * sizeof(float);
    const size_t blocks = size_t(g->N) * g->C * bands;
    if (lds <= 48 * 1024 && blocks < 0x7fffffffu && g->W <= 2048) {
      auto kern = k_pool_max_bwd_tiled<0, 0, 0, 0, S>;
      if (g->kernel_h == 3 && g->kernel_w == 3 && g->stride_h == 2 && g->stride_w == 2)
        kern = k_pool_max_bwd_tiled<3, 3, 2, 2, S>;
      else if (g->kernel_h == 2 && g->kernel_w == 2 && g->stride_h == 2 && g->stride_w == 2)
        kern = k_pool_max_bwd_tiled<2, 2, 2, 2, S>;
      else if (g->kernel_h == 3 && g->kernel_w == 3 && g->stride_h == 1 && g->stride_w == 1)
        kern = k_pool_max_bwd_tiled<3, 3, 1, 1, S>;
      SGH_LAUNCH_TIMED(kern, dim3((unsigned)blocks), dim3(kBlock), lds, sgh_stream_of(stream), dy, x, dx, to_g(g), TH,
                         bands, max_xrows, max_np);
    } else {
      SGH_LAUNCH_TIMED(k_pool_max_bwd<S>, dim3(grid_for(total)), dim3(kBlock), 0, sgh_stream_of(stream), dy, x, dx,
                         to_g(g), total);
    }
  } else if (g->P == 1 && g->Q == 1 && g->pad_h == 0 && g->pad_w == 0 && g->kernel_h >= g->H && g->kernel_w >= g->W &&
             sgh_aligned16(dx))
    SGH_LAUNCH_TIMED(k_pool_avg_bwd_global<S>, dim3(grid_for((total + S::VEC - 1) / S::VEC)), dim3(kBlock), 0,
                       sgh_stream_of(stream), dy, dx, g->H * g->W, total);
  else
    SGH_LAUNCH_TIMED(k_pool_avg_bwd<S>, dim3(grid_for(total)), dim3(kBlock), 0, sgh_stream_of(stream), dy, dx, to_g(g),
                       total);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}

}  // namespace

extern "C" {

int sgh_pool_geom_init(sgh_pool_geom *g, int N, int C, int H, int W, int kernel_h, int kernel_w, int stride_h,
                       int stride_w, int pad_h, int pad_w, int is_max) {
  if (!g) return SGH_EINVAL;
  if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || kernel_h <= 0 || kernel_w <= 0 || stride_h <= 0 || stride_w <= 0 ||
      pad_h < 0 || pad_w < 0)
    return SGH_EINVAL;
  if (H + 2 * pad_h < kernel_h || W + 2 * pad_w < kernel_w) return SGH_EINVAL;
  g->N = N;
  g->C = C;
  g->H = H;
  g->W = W;
  g->kernel_h = kernel_h;
  g->kernel_w = kernel_w;
  g->stride_h = stride_h;
  g->stride_w = stride_w;
  g->pad_h = pad_h;
  g->pad_w = pad_w;
  // PoolingHandle's floor formula (reference: src/model/operation/pooling.cc:48-51)
  g->P = (H + 2 * pad_h - kernel_h) / stride_h + 1;
  g->Q = (W + 2 * pad_w - kernel_w) / stride_w + 1;
  g->is_max = is_max ? 1 : 0;
  return geom_ok(g) ? SGH_OK : SGH_EINVAL;
}

int sgh_pool_fwd_f32(const sgh_pool_geom *g, const float *x, float *y, void *stream) {
  return pool_fwd<StF32>(g, x, y, stream);
}
int sgh_pool_fwd_f16(const sgh_pool_geom *g, const uint16_t *x, uint16_t *y, void *stream) {
  return pool_fwd<StF16>(g, x, y, stream);
}
int sgh_pool_fwd_bf16(const sgh_pool_geom *g, const uint16_t *x, uint16_t *y, void *stream) {
  return pool_fwd<StBF16>(g, x, y, stream);
}
int sgh_pool_relu_fwd_f32(const sgh_pool_geom *g, const float *x, float *y, void *stream) {
  if (!geom_ok(g) || !x || !y) return SGH_EINVAL;
  QuadG qg;
  if (!g->is_max || !quad_plan(g, 4, false, &qg)) return SGH_EUNSUPPORTED;
  hipLaunchKernelGGL((k_pool_quad_fwd<StF32, kQuadReluMax>), dim3(grid_for((size_t(qg.total) + 3) / 4)), dim3(kBlock), 0,
                     sgh_stream_of(stream), x, y, qg);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}
int sgh_pool_relu_bwd_f32(const sgh_pool_geom *g, const float *dy, const float *x, float *dx, void *stream) {
  if (!geom_ok(g) || !dy || !x || !dx) return SGH_EINVAL;
  QuadG qg;
  if (!g->is_max || !quad_plan(g, 4, true, &qg)) return SGH_EUNSUPPORTED;
  hipLaunchKernelGGL((k_pool_quad_bwd<StF32, kQuadReluMax>), dim3(grid_for((size_t(qg.total) + 3) / 4)), dim3(kBlock), 0,
                     sgh_stream_of(stream), dy, x, dx, qg, (g->H + 1) / 2, unsigned(size_t(g->N) * g->C * g->P * g->Q * 4));
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}
int sgh_pool_bwd_f32(const sgh_pool_geom *g, const float *dy, const float *x, const float *y, float *dx,
                     void *stream) {
  return pool_bwd<StF32>(g, dy, x, y, dx, stream);
}
int sgh_pool_bwd_f16(const sgh_pool_geom *g, const uint16_t *dy, const uint16_t *x, const uint16_t *y, uint16_t *dx,
                     void *stream) {
  return pool_bwd<StF16>(g, dy, x, y, dx, stream);
}
int sgh_pool_bwd_bf16(const sgh_pool_geom *g, const uint16_t *dy, const uint16_t *x, const uint16_t *y, uint16_t *dx,
                      void *stream) {
  return pool_bwd<StBF16>(g, dy, x, y, dx, stream);
}

}  // extern "C"
