// fp32 weight gradient of 3x3 convolutions of stride 1 or 2 and padding 1 on the bfloat16 matrix instructions: three parts per value,
// six products (conv_split.hip says why that is fp32 arithmetic).
//
//   dW[k][c][r][s] = sum_{n,p,q} dy[n][k][p][q] * x[n][c][p + r - 1][q + s - 1]
//
// The reduction runs over pixels: a matrix operand holds octets of eight consecutive pixels of a row.  An octet of dy meets the
// x octets of three rows as they are (s = 1) and shifted by one pixel (s = 0, 2): a lane reads the aligned octet and the
// neighbour dword on either side and forms both shifts with funnel shifts, so x is staged once for all nine taps.
//
// A workgroup owns 64 x 64 (k, c) pairs and all nine taps: a wavefront 32 x 32 pairs, 144 accumulators.  Its 512 threads are two
// groups of 2 x 2 wavefronts, each walking half of the workgroup's rows with LDS of its own; the sums meet in LDS at the end, so
// that one partial image per CU goes through memory.  A group walks a strip of up to 32 columns down the images, in "virtual"
// rows (an image is its P rows and a row of zeros): per iteration RPI new rows of dy and of x are fetched into registers while
// the previous ones are multiplied, then split and written; x rows live in a ring of RPI + 2.  Rows of OCS octets (one, two or
// four): the columns beyond Q are zeros on both sides.
//
// Stride 2: the octet's columns 2 q + s - 1 of x are kept apart, the odd ones (s = 2 as they are, s = 0 shifted by one pixel) and the
// even ones (s = 1), and two rows of x come in for one of dy.  That is four times the LDS per pixel, so the strips are half as wide and
// an iteration half as long.  64 images, whole calls, k_wgrad3x3 and this: 64 channels of 56 x 56 to 128 95 -> 85 us, 128 of 28 x 28 to
// 256 95 -> 85, 256 of 14 x 14 to 512 90 -> 89; what that kernel leaves to the generic one: 45 images of 224, 50 x 59, to 213
// 542 -> 314, 17 of 109, 96 x 112, to 268 606 -> 298; 0.3 to 0.45 times the error.  (128 x 32 pairs, with iterations as long as at stride 1:
// eleven registers spilled, 88 to 93 us.)
//
// The sums of the workgroups of a (k, c) tile are added in ascending order by k_wgrad_oct_reduce.
//
// 64 images, whole calls, k_wgrad3x3 and this: 64 channels of 56 x 56 153 -> 105 us, 128 of 28 x 28 133 -> 102, 256 of 14 x 14
// 134 -> 101, 512 of 7 x 7 137 -> 108, with 0.25 to 0.75 times the error against float64.  A tap's six products are summed on their
// own and added to the accumulator once; without that the error is up to 1.5 times that of the fp32 instructions behind a
// ReLU (whose zeros cost those no rounding), and the kernel 7 per cent faster.
#include "common.h"
#include "split_parts.h"

namespace {

constexpr int NT = 512, GT = 256;   // threads of a workgroup, of a group
constexpr int PARTS = 3;
constexpr int kOOB = int(0x80000000u);
constexpr int kAcc = 9 * 16 * 64;   // accumulators of a wavefront

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

struct WoArgs {
  const float *dy, *x;
  float *partial;   // [split][tile][wavefront][accumulator][lane]
  int N, C, K, P, Q, H, W;
  int ktiles, tiles, splits, strips, iters, per_split;   // iterations of a strip, of a workgroup
  unsigned dy_bytes, x_bytes;
};

// E elements of a tensor row as they come from memory: eight, or the sixteen that an octet of dy meets at stride 2
template <int E>
struct Run {
  v4u raw[E / 4];
  int nv;   // valid elements
  // elements [off, off + nv) of the tensor; nothing beyond its last byte is touched
  __device__ __forceinline__ void load(rsrc_t r, unsigned bytes, int off, int nv_) {
    nv = nv_;
    const int at = nv > 0 ? off * 4 : kOOB;
    const bool tail = nv > 0 && unsigned(at) + E * 4 > bytes;
#pragma unroll
    for (int i = 0; i < E / 4; ++i)
      raw[i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, tail ? kOOB : at, 16 * i, 0));
    if (__any(tail)) {
      if (tail) {
#pragma unroll
        for (int j = 0; j < E; ++j) raw[j / 4][j % 4] = __builtin_amdgcn_raw_buffer_load_b32(r, j < nv ? at + 4 * j : kOOB, 0, 0);
      }
    }
  }
  // an octet from element `from` on, every E / 8
  __device__ __forceinline__ void parts(v4u (&out)[PARTS], int from = 0) const {
    constexpr int EVERY = E / 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ia = from + 2 * i * EVERY, ib = ia + EVERY;
      const unsigned ua = raw[ia / 4][ia % 4], ub = raw[ib / 4][ib % 4];
      const float a = ia < nv ? __builtin_bit_cast(float, ua) : 0.f;
      const float b = ib < nv ? __builtin_bit_cast(float, ub) : 0.f;
      const Parts s = split2(a, b);
      out[0][i] = s.p[0], out[1][i] = s.p[1], out[2][i] = s.p[2];
    }
  }
};

template <int OCS, int RPI, int ST>
struct Shape {
  static constexpr int OPI = OCS * RPI, RING = ST == 1 ? RPI + 2 : 2 * RPI + 1;
  // 16-byte units of a channel's x row: the octets, a dword on either side, odd
  // (stride 2: a dword, the octets of the odd columns, those of the even ones)
  static constexpr int XP = ST == 2 ? 2 * OCS + 1 : OCS == 4 ? 7 : OCS == 1 ? 3 : 5;
  static constexpr int XPART = 64 * XP * 16, XROW = PARTS * XPART;
  static constexpr int DYO = (PARTS * 64 + 4) * 16;            // an octet of dy; four units of padding spread the writes over the banks
  static constexpr int GROUP = RING * XROW + OPI * DYO;
  static constexpr int LDS = 2 * GROUP > kAcc * 16 ? 2 * GROUP : kAcc * 16;
  static_assert(OPI * ST == 4 && LDS + 16 <= 160 * 1024, "");
};

template <int OCS, int RPI, int ST>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_wgrad_oct(WoArgs a) {
  typedef Shape<OCS, RPI, ST> S;
  typedef Run<8> Octet;
  typedef Run<8 * ST> XRun;
  constexpr int OPI = S::OPI, RING = S::RING, XO = 4;
  static_assert(ST * OPI == XO && XO * 64 == GT, "an octet of x, or a run of sixteen, per thread; of dy one for all or half of them");
  // elements beside the strip: on either side, or (stride 2) on the left of twice as many rows
  constexpr int EDGE = RPI * 128, EDGES = OCS >= 4 / ST ? 1 : 0;
  static_assert(EDGES * EDGE <= GT, "");
  extern __shared__ __align__(16) char smem[];
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), group = wave >> 2, w4 = wave & 3, wm = w4 >> 1, wn = w4 & 1;
  const int tg = t & (GT - 1);
  char *const xs = smem + group * S::GROUP, *const dys = xs + RING * S::XROW;
  // (the tiles of a split read the same rows: they go to one XCD, as in conv16.hip)
  int tile, split;
  if ((a.splits & 7) == 0) {
    const int slot = int(blockIdx.x) >> 3;
    tile = slot % a.tiles, split = slot / a.tiles * 8 + (int(blockIdx.x) & 7);
  } else {
    tile = int(blockIdx.x) % a.tiles, split = int(blockIdx.x) / a.tiles;
  }
  const int k0 = tile % a.ktiles * 64, c0 = tile / a.ktiles * 64;
  const int strip = split % a.strips, q0 = strip * OCS * 8;
  const int first = split / a.strips * a.per_split, last = min(a.iters, first + a.per_split);
  const int mine = (a.per_split + 1) / 2;                    // iterations of a group (a last one may be empty)
  const int it0 = first + group * mine, it1 = min(last, it0 + mine);
  const int VP = a.P + 1, H = ST == 1 ? a.P : a.H, W = ST == 1 ? a.Q : a.W, VX = VP * ST;
  const rsrc_t rdy = make_rsrc(a.dy, a.dy_bytes), rx = make_rsrc(a.x, a.x_bytes);

  for (int i = tg; i < RING * S::XROW / 16; i += GT) reinterpret_cast<v4u *>(xs)[i] = v4u{0u, 0u, 0u, 0u};

  // ---- staging.  A task is an octet of a channel: o = task % OPI (row o / OCS, octet o % OCS), channel task / OPI
  auto row_of = [&](int v, int &n, int &p) {
    n = v < 0 ? -1 : v / VP, p = v < 0 ? a.P : v - n * VP;
  };
  auto count = [&](int n, int p, int c, int channels, int q) {   // valid elements of the octet at column q
    return p < a.P && n >= 0 && n < a.N && c < channels ? max(0, min(8, a.Q - q)) : 0;
  };
  auto row_of_x = [&](int v, int &n, int &p) {
    n = v < 0 ? -1 : v / VX, p = v < 0 ? H : v - n * VX;
  };
  auto count_x = [&](int n, int p, int c, int q) {
    return p < H && n >= 0 && n < a.N && c < a.C ? max(0, min(8 * ST, W - q * ST)) : 0;
  };
  auto put_x = [&](const XRun &o, int slot, int c, int oc) {
    v4u part[PARTS];
#pragma unroll
    for (int odd = ST - 1; odd >= 0; --odd) {
      o.parts(part, odd);
#pragma unroll
      for (int i = 0; i < PARTS; ++i)
        *reinterpret_cast<v4u *>(xs + slot * S::XROW + i * S::XPART + (c * S::XP + 1 + oc + (ST == 2 && !odd ? OCS : 0)) * 16) = part[i];
    }
  };
  // the element left (side 0) and right (side 1) of the strip
  auto edge_off = [&](int n, int p, int c, int side) {
    const int q = side ? q0 + 8 * OCS : q0 * ST - 1;
    const bool ok = p < H && n >= 0 && n < a.N && c0 + c < a.C && q >= 0 && q < W;
    return ok ? (((n * a.C + c0 + c) * H + p) * W + q) * 4 : kOOB;
  };
  auto edge_get = [&](int off) -> unsigned { return __builtin_amdgcn_raw_buffer_load_b32(rx, off, 0, 0); };
  auto put_edge = [&](unsigned raw, int slot, int c, int side) {
    const Parts s = split2(__builtin_bit_cast(float, raw), 0.f);
    const uint16_t part[PARTS] = {uint16_t(s.p[0]), uint16_t(s.p[1]), uint16_t(s.p[2])};
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
      *reinterpret_cast<uint16_t *>(xs + slot * S::XROW + i * S::XPART + c * S::XP * 16 + (side ? 16 + OCS * 16 : 14)) = part[i];
  };

  int dn, dp, xn, xp, en, ep;   // (image, row) of this thread's next octets and edge
  const int v0 = it0 * RPI;
  // this thread's element of the edges: its row among the new ones, channel, side
  const int edge_row = ST == 1 ? tg >> 7 : tg >> 6, edge_channel = ST == 1 ? tg >> 1 & 63 : tg & 63, edge_side = ST == 1 ? tg & 1 : 0;
  const int first_x = ST == 1 ? v0 + 1 : 2 * v0;
  row_of(v0 + tg % OPI / OCS, dn, dp);
  row_of_x(first_x + tg % XO / OCS, xn, xp);
  row_of_x(first_x + edge_row, en, ep);

  Octet sd;
  XRun sx;
  unsigned se;
  auto step_row = [&](int &n, int &p) {
    p += RPI;
    if (p >= VP) p -= VP, ++n;
  };
  auto step_row_x = [&](int &n, int &p) {
    p += RPI * ST;
    if (p >= VX) p -= VX, ++n;
  };
  // dy rows [v0, v0 + RPI) and x rows [v0 + 1, v0 + RPI], or [2 v0, 2 (v0 + RPI)), of an iteration, then on to the next one
  auto load = [&]() {
    const int k = tg / OPI, c = tg / XO, q = q0 + tg % OCS * 8;
    sd.load(rdy, a.dy_bytes, ((dn * a.K + k0 + k) * a.P + dp) * a.Q + q, k < 64 ? count(dn, dp, k0 + k, a.K, q) : 0);
    sx.load(rx, a.x_bytes, ((xn * a.C + c0 + c) * H + xp) * W + q * ST, count_x(xn, xp, c0 + c, q));
    step_row(dn, dp), step_row_x(xn, xp);
    if (EDGES) {
      se = edge_get(edge_off(en, ep, edge_channel, edge_side));
      step_row_x(en, ep);
    }
  };
  // Every other step's dy is negated, and the other ones in the second group, and what they give is subtracted: the matrix
  // instructions round towards minus infinity on average, which adds up over a sum (1024 channels of 14 x 14, forward pass:
  // 2e-7 of the mean magnitude with one sign, 2e-8 with two).  Stride 2, where an iteration is one step: every other iteration's, and
  // the other way round in every other split, which often is the same rows of another image (64 images, 64 channels of 56 x 56 to 128:
  // the groups alone left 4.0e-8)
  const bool turned = (group != 0) != (ST == 2 && (split / a.strips & 1));
  const unsigned sign = turned ? 0x80008000u : 0u;
  auto slot_of = [](int base, int j) { return base + j < RING ? base + j : base + j - RING; };
  auto stage = [&](int base, int i) {   // of iteration i; base: the ring slot of row v0 - 1, or 2 v0 - 1
    const int o = tg % OPI, k = tg / OPI;
    v4u part[PARTS];
    sd.parts(part);
    if (ST == 1 || k < 64) {
#pragma unroll
      for (int j = 0; j < PARTS; ++j) *reinterpret_cast<v4u *>(dys + o * S::DYO + (j * 64 + k) * 16) = part[j] ^ ((ST == 1 ? o & 2 : i & 1) ? ~sign & 0x80008000u : sign);
    }
    put_x(sx, slot_of(base, 3 - ST + tg % XO / OCS), tg / XO, tg % OCS);
    if (EDGES && (EDGE % GT == 0 || tg < EDGE)) put_edge(se, slot_of(base, 3 - ST + edge_row), edge_channel, edge_side);
  };

  v16f acc[9];
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;

  // rows v0 - 1 and v0, or row 2 v0 - 1, then the first iteration's own
  constexpr int AHEAD = 3 - ST;
  int base = v0 % RING;
  __syncthreads();   // (the zeros are in place)
  for (int i = tg; i < AHEAD * OCS * 64; i += GT) {
    const int oc = i % OCS, c = i / OCS & 63, j = i / (OCS * 64), q = q0 + oc * 8;
    int n, p;
    row_of_x(v0 * ST - 1 + j, n, p);
    XRun o;
    o.load(rx, a.x_bytes, ((n * a.C + c0 + c) * H + p) * W + q * ST, count_x(n, p, c0 + c, q));
    put_x(o, slot_of(base, j), c, oc);
  }
  if (EDGES && edge_row < AHEAD) {
    int n, p;
    row_of_x(v0 * ST - 1 + edge_row, n, p);
    put_edge(edge_get(edge_off(n, p, edge_channel, edge_side)), slot_of(base, edge_row), edge_channel, edge_side);
  }
  load();
  stage(base, 0);
  __syncthreads();

  const char *const da = dys + half * S::DYO + (wm * 32 + l32) * 16;
  const char *const xb = xs + (wn * 32 + l32) * S::XP * 16 + 12;
  for (int i = 0; i < mine; ++i) {
    const bool more = i + 1 < mine;
    if (more) load();
    if (it0 + i < it1) {
      [[maybe_unused]] const float turn = i & 1 ? -1.f : 1.f;
      struct Raw {
        v4u d, e;        // (stride 2: of the odd columns and of the even ones)
        unsigned l, r;
      };
      // unit u = (step, row r of the filter): the three parts of the octet and its neighbours, three taps.  A tap's six products
      // are summed on their own, the small ones first, and the sum is added to the accumulator: one rounding there for 16
      // pixels instead of six or more.  A part of the next unit is read as soon as the last tap has taken its own.
      constexpr int UNITS = OPI / 2 * 3;
      auto read = [&](int u, int p) {
        const int s = u / 3, r = u % 3, oa = 2 * s, ob = 2 * s + 1;
        const int ja = slot_of(base, oa / OCS * ST + r) * S::XROW + oa % OCS * 16;
        const int jb = slot_of(base, ob / OCS * ST + r) * S::XROW + ob % OCS * 16;
        const char *at = xb + (half ? jb : ja) + p * S::XPART;
        Raw w;
        w.l = *reinterpret_cast<const unsigned *>(at);
        w.d = *reinterpret_cast<const v4u *>(at + 4);
        if (ST == 1) w.r = *reinterpret_cast<const unsigned *>(at + 20);
        else w.e = *reinterpret_cast<const v4u *>(at + 4 + OCS * 16);
        return w;
      };
      v4u A[PARTS];
      auto read_a = [&](int s) {
#pragma unroll
        for (int p = PARTS - 1; p >= 0; --p) A[p] = *reinterpret_cast<const v4u *>(da + 2 * s * S::DYO + p * 1024);
      };
      Raw w[PARTS];
      read_a(0);
#pragma unroll
      for (int p = PARTS - 1; p >= 0; --p) w[p] = read(0, p);
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        const int s = u / 3, r = u % 3;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          v16f sum;
#pragma unroll
          for (int v = 0; v < 16; ++v) sum[v] = 0.f;
#pragma unroll
          for (int p = PARTS - 1; p >= 0; --p) {
            const v4u d = w[p].d;
            v4u x = ST == 2 && c == 1 ? w[p].e : d;   // (stride 2: columns 2 q - 1, 2 q, 2 q + 1)
            if (ST == 1 ? c != 1 : c == 0) {
              const unsigned m1 = __builtin_amdgcn_alignbit(d[1], d[0], 16), m2 = __builtin_amdgcn_alignbit(d[2], d[1], 16),
                             m3 = __builtin_amdgcn_alignbit(d[3], d[2], 16);
              if (c == 0) x = v4u{__builtin_amdgcn_alignbit(d[0], w[p].l, 16), m1, m2, m3};
              else x = v4u{m1, m2, m3, __builtin_amdgcn_alignbit(w[p].r, d[3], 16)};
            }
            if (c == 2 && u + 1 < UNITS) w[p] = read(u + 1, p);
#pragma unroll
            for (int q = PARTS - 1 - p; q >= 0; --q) sum = mfma(A[q], x, sum);
          }
          if (r == 2 && c == 2 && s + 1 < OPI / 2) read_a(s + 1);
          v16f &total = acc[r * 3 + c];
          if constexpr (ST == 1) total = s % 2 ? total - sum : total + sum;
          else
#pragma unroll
            for (int v = 0; v < 16; ++v) total[v] = __builtin_fmaf(sum[v], turn, total[v]);
          asm volatile("" : "+v"(total));   // (here, not when all taps' sums are there)
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    __syncthreads();
    if (more) {
      base = slot_of(base, RPI * ST);
      stage(base, i + 1);
      __syncthreads();
    }
  }

  // ---- sums that are not finite: an infinity or a value too large for the scale has parts whose products are NaN, and a zero of
  // the virtual rows and columns has met one.  All of the workgroup's sums are formed again on the fp32 instructions, a row at a
  // time, whatever the values are: 2.7 times the products' time.  (LDS is free.  Everything is derived anew from opaque copies:
  // what the loop above holds in registers for this, it spills.)
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] *= kSplitUnscale, bad |= !finite(acc[i][v]);
  int *const again = reinterpret_cast<int *>(smem);
  if (t == 0) *again = 0;
  __syncthreads();
  if (__any(bad) && lane == 0) *again = 1;
  __syncthreads();
  if (*again) {
    constexpr int COLS = 8 * OCS, YP = COLS + 1, XW = ST == 1 ? COLS + 2 : 2 * COLS + 1, XF = XW | 1;   // odd pitches
    static_assert((64 * YP + 192 * XF) * 4 <= S::GROUP, "");
    int tt = threadIdx.x, P = a.P, Q = a.Q, H = ST == 1 ? P : a.H, W = ST == 1 ? Q : a.W;
    asm volatile("" : "+v"(tt), "+s"(P), "+s"(Q), "+s"(H), "+s"(W));
    const int th = tt >> 5 & 1, row = wm * 32 + (tt & 31), col = wn * 32 + (tt & 31);
    float *const ys = reinterpret_cast<float *>(smem + group * S::GROUP), *const xr = ys + 64 * YP;
    unsigned valid = 0;   // accumulator registers that hold a filter
#pragma unroll
    for (int v = 0; v < 16; ++v) valid |= unsigned(k0 + wm * 32 + 8 * (v >> 2) + 4 * th + (v & 3) < a.K && c0 + col < a.C) << v;
    // not every sum of this wavefront, of the workgroup is a NaN yet (in a diverged network they soon are)
    bool number = true;
    int *const numbers = reinterpret_cast<int *>(smem + S::LDS);   // the last row that left one
    if (tt == 0) *numbers = -1;
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
    for (int i = 0; i < mine * RPI; ++i) {
      const int v = it0 * RPI + i, n = v / (P + 1), p = v - n * (P + 1);
      const bool live = v < it1 * RPI && n < a.N && p < P;
      __syncthreads();
      if (*numbers < i - 1) break;
      if (live) {
        for (int e = tt & (GT - 1); e < 64 * COLS; e += GT) {
          const int ch = e / COLS, q = e % COLS;
          ys[ch * YP + q] = k0 + ch < a.K && q0 + q < Q ? a.dy[((n * a.K + k0 + ch) * P + p) * Q + q0 + q] : 0.f;
        }
        for (int e = tt & (GT - 1); e < 192 * XW; e += GT) {
          const int ch = e / XW % 64, h = p * ST + e / (XW * 64) - 1, w = q0 * ST + e % XW - 1;
          const bool in = c0 + ch < a.C && unsigned(h) < unsigned(H) && unsigned(w) < unsigned(W);
          xr[e / XW * XF + e % XW] = in ? a.x[((n * a.C + c0 + ch) * H + h) * W + w] : 0.f;
        }
      }
      __syncthreads();
      if (live && number) {
#pragma unroll 1
        for (int u = 0; u < COLS; u += 2) {
          const float d = ys[row * YP + u + th];
          const bool in = q0 + u + th < Q;   // (beyond the row dy's zeros must meet zeros)
#pragma unroll
          for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const float xv = xr[(r * 64 + col) * XF + (u + th) * ST + c];
              acc[r * 3 + c] = __builtin_amdgcn_mfma_f32_32x32x2f32(d, in ? xv : 0.f, acc[r * 3 + c], 0, 0, 0);
            }
        }
        bool any = false;
#pragma unroll
        for (int c = 0; c < 9; ++c)
#pragma unroll
          for (int u = 0; u < 16; ++u) any |= acc[c][u] == acc[c][u] && (valid >> u & 1);
        number = __any(any);
      }
      if (number && lane == 0) *numbers = i;
    }
    if (turned) {   // (as the loop above leaves it)
#pragma unroll
      for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = -acc[i][v];
    }
    __syncthreads();
  }

  // ---- the two groups' sums, then this workgroup's partial image
  float *const ex = reinterpret_cast<float *>(smem) + w4 * kAcc + lane;
  if (group) {
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) ex[(i * 16 + v) * 64] = acc[i][v];
  }
  __syncthreads();
  if (group) return;
  const rsrc_t rp = make_rsrc(a.partial + (size_t(split) * a.tiles + tile) * 4 * kAcc, 4 * kAcc * 4);
  const int po = (w4 * kAcc + lane) * 4;
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, acc[i][v] - ex[(i * 16 + v) * 64]) ^ (sign & 0x80000000u), rp, po, (i * 16 + v) * 256, 0);
}

// dW from the partial images, in ascending order.  A workgroup takes four accumulator registers of a wavefront (16 bytes a lane:
// 4 bytes a lane and one register a workgroup read the 38 MB of a layer in 12 us, this in 9) and nine taps: stretches of 288
// weights; ZL threads share the images of a sum, ZL workgroups the taps.
template <int ZL>
__global__ __launch_bounds__(576) void k_wgrad_oct_reduce(WoArgs a, float *__restrict__ dW) {
  constexpr int TAPS = 9 / ZL;   // taps of a workgroup
  typedef float v4f __attribute__((ext_vector_type(4)));
  __shared__ double sums[ZL][TAPS][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, z = wave / TAPS, ti = wave % TAPS;
  const int tap0 = int(blockIdx.x) % ZL * TAPS, b = int(blockIdx.x) / ZL, v = b % 4 * 4, w4 = b / 4 % 4, tile = b / 16;
  const size_t image = size_t(a.tiles) * 4 * kAcc;
  const float *p = a.partial + (size_t(tile) * 4 + w4) * kAcc + ((tap0 + ti) * 16 + v) * 64 + lane * 4;
  double s[4] = {0, 0, 0, 0};   // (in fp32 256 images add a tenth to the error of their sums)
#pragma unroll 4
  for (int i = z; i < a.splits; i += ZL) {
    const v4f x = *reinterpret_cast<const v4f *>(p + i * image);
#pragma unroll
    for (int d = 0; d < 4; ++d) s[d] += x[d];
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) sums[z][ti][lane * 4 + d] = s[d];
  __syncthreads();
  for (int e = threadIdx.x; e < TAPS * 256; e += 576) {
    const int l = e / TAPS, tj = e % TAPS;   // l: register, lane of an accumulator
    double r = sums[0][tj][l];
#pragma unroll
    for (int i = 1; i < ZL; ++i) r += sums[i][tj][l];
    const int k = tile % a.ktiles * 64 + (w4 >> 1) * 32 + 2 * v + 4 * (l >> 5 & 1) + (l >> 6);
    const int c = tile / a.ktiles * 64 + (w4 & 1) * 32 + (l & 31);
    if (k < a.K && c < a.C) dW[(size_t(k) * a.C + c) * 9 + tap0 + tj] = float(r);
  }
}

struct WoPlan {
  bool ok;
  int st, ocs, rpi, ktiles, tiles, splits, strips, iters, per_split;
};

// Expected us of a plan of stride 2 (fitted over 96 layers): 3.6 for an iteration of either group, 0.06 for an image written and summed
double expected_us(const WoPlan &p) {
  const long wgs = long(p.tiles) * p.splits, cus = sgh_num_cus();
  return 6 + double((wgs + cus - 1) / cus) * ((p.per_split + 1) / 2) * 3.6 + 0.06 * double(wgs);
}

size_t image_bytes(const WoPlan &p) { return size_t(p.splits) * p.tiles * 4 * kAcc * sizeof(float); }

// `room`: bytes for the partial images
WoPlan plan(const sgh_conv_geom *g, size_t room) {
  WoPlan p{};
  p.st = g->stride_h;
  if (g->R != 3 || g->S != 3 || p.st < 1 || p.st > 2 || g->stride_w != p.st || g->pad_h != 1 || g->pad_w != 1) return p;
  if (g->P != (g->H + p.st - 1) / p.st || g->Q != (g->W + p.st - 1) / p.st) return p;
  const size_t pixels = size_t(g->N) * g->P * g->Q, lim = size_t(1) << 29;
  if (size_t(g->N) * g->H * g->W * g->C >= lim || pixels * g->K >= lim) return p;
  // Few channels leave the 64 columns of a tile empty (their nine taps are columns to the fp32 kernels: 3, 11 and 25 of 64
  // channels 0.6 times as fast, 39 and more 1.1 to 2.4 times).  Below 0.7 G products a launch is short beside its partial images:
  // 0.13 to 0.67 G, 55 layers, 0.9 to 1.5 times as fast, and the rule that would tell those apart is not there.
  if (20 * g->C < 11 * 64 * ((g->C + 63) / 64) || double(pixels) * g->K * g->C * 9 < 7e8) return p;
  const int oc = (g->Q + 7) / 8, widest = 4 / p.st;   // (stride 2: twice the columns of x)
  p.strips = (oc + widest - 1) / widest;
  p.ocs = (oc + p.strips - 1) / p.strips;
  if (p.ocs == 3) p.ocs = 4;   // (two rows of three octets do not fit the registers: 64 images, 96 channels of 20 x 22 109 against 102 us)
  p.rpi = widest / p.ocs;
  if (g->P + 1 < p.rpi || size_t(g->N) * (g->P + 1) >= (size_t(1) << 30)) return p;
  p.iters = int((size_t(g->N) * (g->P + 1) + p.rpi - 1) / p.rpi);
  p.ktiles = (g->K + 63) / 64;
  const long tiles = long(p.ktiles) * ((g->C + 63) / 64);
  if (tiles > 65536) return p;
  p.tiles = int(tiles);
  const int cus = sgh_num_cus();
  // one workgroup per CU, two iterations at least for either of its groups
  const long most = p.iters / 4 > 0 ? p.iters / 4 : 1;
  auto split = [&](long sp) {
    if (sp > most) sp = most;
    if (sp < 1) sp = 1;
    p.per_split = int((p.iters + sp - 1) / sp);
    p.splits = (p.iters + p.per_split - 1) / p.per_split * p.strips;
  };
  const long one = cus / (tiles * p.strips);
  split(one);
  // Stride 2, more than a quarter as many tiles and strips as CUs: one to three splits of them leave up to half of the CUs idle in their only or
  // last round.  Up to three rounds of shorter workgroups do not, if there is room for their images: 35 images, 654 channels of 31 x 36 to 344,
  // 132 workgroups 1017 us, 660 of them 661 (k_wgrad3x3 766); 7 of 811, 73 x 70, to 488 980 -> 751 (the generic kernel 887); 4 of 299, 88 x 107,
  // to 417 344 -> 258.
  if (p.st == 2 && one < 4) {
    WoPlan best = p;
    double least = expected_us(p);
    for (long sp = one + 1; sp * tiles * p.strips <= 3l * cus && sp <= most; ++sp) {
      split(sp);
      if (const double us = expected_us(p); us < least && image_bytes(p) <= room) least = us, best = p;
    }
    p = best;
  }
  p.ok = true;
  return p;
}

template <int OCS, int RPI, int ST>
int launch(const WoArgs &a, hipStream_t s) {
  auto kern = k_wgrad_oct<OCS, RPI, ST>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) !=
        hipSuccess)
      return SGH_EUNSUPPORTED;
    attr_set = true;
  }
  SGH_LAUNCH_TIMED(kern, dim3(unsigned(a.tiles * a.splits)), dim3(NT), (Shape<OCS, RPI, ST>::LDS + 16), s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

}  // namespace

size_t sgh_wgrad_oct_workspace_bytes(const sgh_conv_geom *g, bool least) {
  const WoPlan p = plan(g, least ? 0 : size_t(-1));
  return p.ok && !sgh_env().conv_split_off ? image_bytes(p) : 0;
}

double sgh_wgrad_oct_us(const sgh_conv_geom *g) { return expected_us(plan(g, size_t(-1))); }

int sgh_wgrad_oct_run(const sgh_conv_geom *g, const float *dy, const float *x, float *dW, void *workspace, size_t ws_bytes,
                      hipStream_t s) {
  const WoPlan p = plan(g, ws_bytes);
  if (!p.ok) return SGH_EUNSUPPORTED;
  WoArgs a;
  a.dy = dy, a.x = x, a.partial = static_cast<float *>(workspace);
  a.N = g->N, a.C = g->C, a.K = g->K, a.P = g->P, a.Q = g->Q, a.H = g->H, a.W = g->W;
  a.ktiles = p.ktiles, a.tiles = p.tiles, a.splits = p.splits, a.strips = p.strips, a.iters = p.iters, a.per_split = p.per_split;
  const size_t pixels = size_t(g->N) * g->P * g->Q;
  a.dy_bytes = unsigned(pixels * g->K * 4), a.x_bytes = unsigned(size_t(g->N) * g->H * g->W * g->C * 4);
  sgh_prof_kernel_begin("conv_wgrad/k_wgrad_oct", 2.0 * pixels * g->K * g->C * 9);
  const int rc = p.ocs == 4   ? launch<4, 1, 1>(a, s)
                 : p.ocs == 2 ? (p.st == 1 ? launch<2, 2, 1>(a, s) : launch<2, 1, 2>(a, s))
                              : (p.st == 1 ? launch<1, 4, 1>(a, s) : launch<1, 2, 2>(a, s));
  sgh_prof_kernel_end(s);
  if (rc != SGH_OK) return rc;
  // (threads per accumulator: as many as leave each a few images)
  const unsigned blocks = unsigned(a.tiles) * 16;
  if (a.splits >= 24) hipLaunchKernelGGL(k_wgrad_oct_reduce<9>, dim3(blocks * 9), dim3(576), 0, s, a, dW);
  else if (a.splits >= 6) hipLaunchKernelGGL(k_wgrad_oct_reduce<3>, dim3(blocks * 3), dim3(576), 0, s, a, dW);
  else hipLaunchKernelGGL(k_wgrad_oct_reduce<1>, dim3(blocks), dim3(576), 0, s, a, dW);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}
