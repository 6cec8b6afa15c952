// 16-bit weight gradient of 3x3 convolutions of padding 1 and stride 1 or 2 (reference: GpuConvBackwardW,
// src/model/operation/convolution.cc:634-681 on half tensors), all nine taps of a pair of channel tiles in one workgroup.
//
//   dW[k][c][r][s] = sum_{n,p,q} dy[n][k][p][q] * x[n][c][st p + r - 1][st q + s - 1]
//
// A matrix operand holds octets of eight consecutive pixels of a row.  k_wgrad16 loads an x octet per tap, nine times the tensor;
// here x is staged once and the taps of a row come from one read of LDS:
//   stride 1: the aligned octet and the neighbour dword on either side, shifted by one pixel with funnel shifts;
//   stride 2: a row is kept as its even and its odd columns; tap 1 is the even octet, tap 2 the odd one, tap 0 the odd one shifted.
//
// A workgroup owns 64 x 64 (k, c) pairs: a wavefront 32 x 32 of them, 144 accumulators.  Its 512 threads are two groups of 2 x 2
// wavefronts, each walking half of the workgroup's rows with LDS of its own; the sums meet in LDS at the end, so that one partial
// image per CU goes through memory.  A group walks a strip of up to 32 output columns down the images in "virtual" rows (an image
// is its P rows and a row of zeros).  Per iteration RPI rows are multiplied, the next RPI are written to LDS (a second buffer of
// dy, a ring of x rows) and the ones after that are requested: one barrier, and a load has an iteration (about 1 us) to arrive.
// The first group stages before it multiplies, the second one after: the two wavefronts of a SIMD are a group each, and one's
// staging arithmetic runs beside the other's matrix instructions.
//
// 128 images f16, with the reduction, k_wgrad16 before and this: stride 1, 64 channels of 56 x 56 89 -> 67 us, 128 of 28 x 28
// 68 -> 59, 256 of 14 x 14 79 -> 54, 512 of 7 x 7 107 -> 59 (500 TFLOP/s); stride 2, 128 of 56 x 56 87 -> 66, 256 of 28 x 28
// 104 -> 64, 512 of 14 x 14 135 -> 70.  Of the 47 us of the kernel the matrix instructions are 16; the rest is LDS reads about as
// long as they are, the staging arithmetic, 5 us in front of the first product and 38 MB of partial images written at once.
#include <type_traits>

#include "common.h"
#include "storage.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

constexpr int NT = 512, GT = 256;   // threads of a workgroup, of a group
constexpr int kOOB = int(0x80000000u);
constexpr int kAcc = 9 * 16 * 64;   // accumulators of a wavefront

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

template <bool BF16>
__device__ __forceinline__ v16f mfma(v4u a, v4u b, v16f c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < __builtin_inff(); }

struct Wo16Args {
  const uint16_t *dy, *x;
  float *partial;   // [split][tile][wavefront][accumulator][lane]
  int N, C, K, H, W, P, Q;
  int ktiles, tiles, ranges, strips, iters, per_range;   // iterations of a strip, of a workgroup
  unsigned dy_bytes, x_bytes;
};

// bits of an octet's first n elements
__device__ __forceinline__ v4u keep_first(int n) {
  v4u m;
#pragma unroll
  for (int d = 0; d < 4; ++d) m[d] = n >= 2 * d + 2 ? ~0u : n == 2 * d + 1 ? 0xffffu : 0u;
  return m;
}

// The eight elements at byte `off` of a tensor, of which the first nv are there (the others are anything); nothing beyond its
// last byte is touched
__device__ __forceinline__ v4u load8(rsrc_t r, unsigned bytes, unsigned off, int nv) {
  const int at = nv > 0 ? int(off) : kOOB;
  const bool tail = nv > 0 && unsigned(at) + 16 > bytes;
  v4u v = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, tail ? kOOB : at, 0, 0));
  if (__any(tail)) {
    if (tail) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned e = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(r, j < nv ? at + 2 * j : kOOB, 0, 0));
        v[j / 2] = j % 2 ? v[j / 2] | e << 16 : e;
      }
    }
  }
  return v;
}

template <int ST, int OCS, int RPI>
struct Shape {
  static constexpr int OPI = OCS * RPI;
  // x rows of a virtual row (stride 2: an even one, an odd one), virtual rows in front of the first that an iteration fetches
  static constexpr int PAR = ST, BEFORE = ST == 1 ? 2 : 1, RING = 2 * RPI + BEFORE;
  // 16-byte units of a channel's x row, an odd number: a dword on the left, the octets and (stride 1) a dword on the right or
  // (stride 2) the octets of the even columns behind those of the odd ones
  static constexpr int XP = ST == 2 ? 2 * OCS + 1 : OCS == 4 ? 7 : OCS == 1 ? 3 : 5;
  static constexpr int XROW = (64 * XP + 4) * 16, XV = PAR * XROW;   // (the padding spreads writes of two rows over the banks)
  static constexpr int DYO = 65 * 16, DYB = OPI * DYO;               // an octet of dy, a buffer of them
  static constexpr int GROUP = RING * XV + 2 * DYB;
  static constexpr int LDS = 2 * GROUP > kAcc * 16 ? 2 * GROUP : kAcc * 16;
  static_assert(OPI % 2 == 0 && XP % 2 == 1 && LDS + 16 <= 160 * 1024, "");
};

template <int ST, int OCS, int RPI, bool BF16>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_wgrad_oct16(Wo16Args a) {
  typedef Shape<ST, OCS, RPI> S;
  constexpr int OPI = S::OPI, RING = S::RING, PAR = S::PAR;
  constexpr int DT = (OPI * 64 + GT - 1) / GT, XT = (OPI * PAR * 64 + GT - 1) / GT;   // octets of dy, (pairs of) octets of x
  constexpr int SIDES = ST == 1 ? 2 : 1, ET = OCS >= 3 ? (RPI * PAR * SIDES * 64 + GT - 1) / GT : 0;
  extern __shared__ __align__(16) char smem[];
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), group = wave >> 2, w4 = wave & 3, wm = w4 >> 1, wn = w4 & 1;
  const int tg = t & (GT - 1);
  char *const xs = smem + group * S::GROUP, *const dys = xs + RING * S::XV;
  // (the tiles and strips of a range of rows read the same lines: they go to one XCD, workgroup w runs on XCD w % 8)
  int tile, strip, range;
  {
    const bool dealt = (a.ranges & 7) == 0;
    const int slot = dealt ? int(blockIdx.x) >> 3 : int(blockIdx.x), rest = slot / a.tiles;
    tile = slot - rest * a.tiles, strip = rest % a.strips;
    range = dealt ? rest / a.strips * 8 + (int(blockIdx.x) & 7) : rest / a.strips;
  }
  const int k0 = tile % a.ktiles * 64, c0 = tile / a.ktiles * 64, q0 = strip * OCS * 8;
  const int first = range * a.per_range, last = min(a.iters, first + a.per_range);
  const int mine = (a.per_range + 1) / 2;                    // iterations of a group (the last ones may be empty)
  const int it0 = first + group * mine, it1 = min(last, it0 + mine);
  const int VP = a.P + 1, PQ = a.P * a.Q, HW = a.H * a.W;
  const rsrc_t rdy = make_rsrc(a.dy, a.dy_bytes), rx = make_rsrc(a.x, a.x_bytes);

  // ---- staging.  An octet of dy is (row j / OCS, octet j % OCS) with j = i % OPI and channel i / OPI, one of x has a row parity
  // between them; its column, channel and masks stay, its row moves on
  auto row_of = [&](int v, int &n, int &p) { n = v < 0 ? -1 : v / VP, p = v < 0 ? a.P : v - n * VP; };
  auto row_ok = [&](int n, int p) { return p < a.P && n >= 0 && n < a.N; };
  auto x_at = [&](int slot, int par, int c) { return xs + slot * S::XV + par * S::XROW + c * S::XP * 16; };
  struct XRaw {
    v4u v[ST];
  };
  // x octet oc of (image n, virtual row p, parity), channel c of the tile
  auto load_x = [&](int n, int p, int par, int c, int oc) {
    const int h = ST * p + par, w = ST * (q0 + oc * 8);
    const bool ok = row_ok(n, p) && h < a.H && c < 64 && c0 + c < a.C;
    const unsigned off = unsigned((n * a.C + c0 + c) * HW + h * a.W + w) * 2;
    XRaw o;
#pragma unroll
    for (int i = 0; i < ST; ++i) o.v[i] = load8(rx, a.x_bytes, off + 16 * i, ok ? a.W - w - 8 * i : 0);
    return o;
  };
  // (m: the octet's elements inside the row, stride 2: of the odd columns and of the even ones)
  auto put_x = [&](const XRaw &o, v4u m, v4u m_even, int slot, int par, int c, int oc) {
    char *const at = x_at(slot, par, c) + (1 + oc) * 16;
    if constexpr (ST == 1) {
      *reinterpret_cast<v4u *>(at) = o.v[0] & m;
    } else {
      v4u even, odd;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned lo = o.v[j / 2][2 * j % 4], hi = o.v[j / 2][2 * j % 4 + 1];
        even[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100), odd[j] = __builtin_amdgcn_perm(hi, lo, 0x07060302);
      }
      *reinterpret_cast<v4u *>(at) = odd & m;
      *reinterpret_cast<v4u *>(at + OCS * 16) = even & m_even;
    }
  };
  // the element left (side 0) and, stride 1, right (side 1) of the strip
  auto load_edge = [&](int n, int p, int par, int c, int side) -> uint16_t {
    const int h = ST * p + par, w = side ? q0 + 8 * OCS : ST * q0 - 1;
    const bool ok = row_ok(n, p) && h < a.H && c0 + c < a.C && w >= 0 && w < a.W;
    return uint16_t(__builtin_amdgcn_raw_buffer_load_b16(rx, ok ? ((n * a.C + c0 + c) * HW + h * a.W + w) * 2 : kOOB, 0, 0));
  };
  auto put_edge = [&](uint16_t v, int slot, int par, int c, int side) {
    *reinterpret_cast<uint16_t *>(x_at(slot, par, c) + (side ? 16 + OCS * 16 : 14)) = v;
  };

  // Requests.  A row of octets steps by RPI virtual rows: a byte offset and a row per octet (octets of a thread that are whole rows
  // of tasks apart share them but for the channel).  Rows behind the last image end beyond the tensor and read as zeros.
  constexpr int XPI = OPI * PAR, DR = GT % OPI == 0 ? 1 : DT, XR = GT % XPI == 0 ? 1 : XT;
  constexpr int AHEAD = ST == 1 ? 1 : 0;   // the virtual row of x that the last row of dy meets
  const int K2 = a.K * PQ * 2, C2 = a.C * HW * 2;
  unsigned dat[DT], xat[XT], eat[ET ? ET : 1];
  int dp[DR], xh[XR], eh[ET ? ET : 1];   // row of dy, row of x (the zeros' rows are P and more, H and more)
  v4u dmask[DR], xmask[ST == 2 ? 2 * XR : 1];
  auto start = [&](int v, int jump, int pitch, int &p) -> unsigned {   // the offset of virtual row v
    const int n = v / VP;
    p = v - n * VP;
    return unsigned(n) * unsigned(jump) + unsigned(p * pitch);
  };
#pragma unroll
  for (int e = 0; e < DT; ++e) {
    const int i = e * GT + tg, ch = i / OPI;
    const unsigned at = start(it0 * RPI + i % OPI / OCS, K2, a.Q * 2, dp[e % DR]) + unsigned((k0 + ch) * PQ + q0 + i % OCS * 8) * 2;
    dat[e] = at;
    dmask[e % DR] = keep_first(a.Q - q0 - i % OCS * 8);
  }
#pragma unroll
  for (int e = 0; e < XT; ++e) {
    const int i = e * GT + tg, c = i / XPI, q = q0 + i % OCS * 8;
    int p;
    const unsigned at = start(it0 * RPI + AHEAD + i % XPI / (OCS * PAR), C2, ST * a.W * 2, p);
    const int par = i / OCS % PAR;
    xat[e] = at + unsigned((c0 + c) * HW + par * a.W + ST * q) * 2;
    xh[e % XR] = ST * p + par;
    if (ST == 2) xmask[e % XR] = keep_first(a.W / 2 - q), xmask[(ST == 2 ? XR : 0) + e % XR] = keep_first((a.W + 1) / 2 - q);
  }
#pragma unroll
  for (int e = 0; e < ET; ++e) {
    const int i = e * GT + tg, side = i % SIDES, c = i / SIDES & 63, par = i / (64 * SIDES) % PAR, w = side ? q0 + 8 * OCS : ST * q0 - 1;
    int p;
    const unsigned at = start(it0 * RPI + AHEAD + i / (64 * SIDES * PAR), C2, ST * a.W * 2, p);
    eat[e] = at + unsigned((c0 + c) * HW + par * a.W + w) * 2;
    eh[e] = c0 + c < a.C && w >= 0 && w < a.W ? ST * p + par : -1;
  }
  // (masks that stay in registers)
#pragma unroll
  for (int e = 0; e < DR; ++e) asm("" : "+v"(dmask[e]));
  if (ST == 2) {
#pragma unroll
    for (int e = 0; e < 2 * XR; ++e) asm("" : "+v"(xmask[ST == 2 ? e : 0]));
  }

  v4u sd[DT];
  XRaw sx[XT];
  uint16_t se[ET ? ET : 1];
  int ahead = it0 * RPI;   // first row of dy of the next request
  auto load = [&]() {   // the rows of an iteration, then on to the next one
    // an octet that crosses the tensor's end lies within eight elements of it, hence in the last image's last rows
    const bool careful = ahead + 2 * RPI + 10 >= a.N * VP;
    ahead += RPI;
    auto request = [&](auto slow) {
#pragma unroll
      for (int e = 0; e < DT; ++e) {
        const int i = e * GT + tg, ch = i / OPI;
        const bool ok = dp[e % DR] < a.P && (OPI * 64 % GT == 0 || ch < 64) && k0 + ch < a.K;
        if constexpr (slow) sd[e] = load8(rdy, a.dy_bytes, dat[e], ok ? a.Q - q0 - i % OCS * 8 : 0);
        else sd[e] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rdy, ok ? int(dat[e]) : kOOB, 0, 0));
      }
#pragma unroll
      for (int e = 0; e < XT; ++e) {
        const int i = e * GT + tg, c = i / XPI;
        const bool ok = xh[e % XR] < a.H && (XPI * 64 % GT == 0 || c < 64) && c0 + c < a.C;
#pragma unroll
        for (int u = 0; u < ST; ++u) {
          if constexpr (slow) sx[e].v[u] = load8(rx, a.x_bytes, xat[e] + 16 * u, ok ? a.W - ST * (q0 + i % OCS * 8) - 8 * u : 0);
          else sx[e].v[u] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rx, ok ? int(xat[e]) : kOOB, 16 * u, 0));
        }
      }
    };
    if (careful) request(std::true_type{});
    else request(std::false_type{});
#pragma unroll
    for (int e = 0; e < ET; ++e)
      se[e] = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(rx, unsigned(eh[e]) < unsigned(a.H) ? int(eat[e]) : kOOB, 0, 0));
    // on to the next iteration's rows
    int dwrap[DR], xwrap[XR];
#pragma unroll
    for (int e = 0; e < DR; ++e) {
      dp[e] += RPI;
      const bool over = dp[e] >= VP;
      dp[e] -= over ? VP : 0;
      dwrap[e] = RPI * a.Q * 2 + (over ? K2 - VP * a.Q * 2 : 0);
    }
#pragma unroll
    for (int e = 0; e < XR; ++e) {
      xh[e] += ST * RPI;
      const bool over = xh[e] >= ST * VP;
      xh[e] -= over ? ST * VP : 0;
      xwrap[e] = ST * RPI * a.W * 2 + (over ? C2 - ST * VP * a.W * 2 : 0);
    }
#pragma unroll
    for (int e = 0; e < DT; ++e) dat[e] += dwrap[e % DR];
#pragma unroll
    for (int e = 0; e < XT; ++e) xat[e] += xwrap[e % XR];
#pragma unroll
    for (int e = 0; e < ET; ++e) {
      if (eh[e] >= 0) {
        eh[e] += ST * RPI;
        const bool over = eh[e] >= ST * VP;
        eh[e] -= over ? ST * VP : 0;
        eat[e] += ST * RPI * a.W * 2 + (over ? C2 - ST * VP * a.W * 2 : 0);
      }
    }
  };
  auto slot_of = [](int base, int j) { return base + j < RING ? base + j : base + j - RING; };
  auto stage = [&](int base, int buffer) {   // base: the ring slot of the row before the iteration's first
    char *const db = dys + buffer * S::DYB;
#pragma unroll
    for (int e = 0; e < DT; ++e) {
      const int i = e * GT + tg, ch = i / OPI;
      if (OPI * 64 % GT == 0 || ch < 64)
        *reinterpret_cast<v4u *>(db + i % OPI * S::DYO + ch * 16) = sd[e] & dmask[e % DR];
    }
#pragma unroll
    for (int e = 0; e < XT; ++e) {
      const int i = e * GT + tg, c = i / (OPI * PAR);
      if (OPI * PAR * 64 % GT == 0 || c < 64)
        put_x(sx[e], ST == 1 ? dmask[e % DR] : xmask[e % XR], xmask[ST == 2 ? XR + e % XR : 0], slot_of(base, S::BEFORE + i % (OPI * PAR) / (OCS * PAR)), i / OCS % PAR, c, i % OCS);
    }
#pragma unroll
    for (int e = 0; e < ET; ++e) {
      const int i = e * GT + tg;
      if (RPI * PAR * SIDES * 64 % GT == 0 || i < RPI * PAR * SIDES * 64)
        put_edge(se[e], slot_of(base, S::BEFORE + i / (64 * SIDES * PAR)), i / (64 * SIDES) % PAR, i / SIDES & 63, i % SIDES);
    }
  };

  v16f acc[9];
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;

  // the rows before those that the first iteration fetches, then its own: all requested before the first is waited for
  constexpr int PT = (S::BEFORE * PAR * OCS * 64 + GT - 1) / GT;
  int base = 0;
  XRaw before[PT];
#pragma unroll
  for (int e = 0; e < PT; ++e) {
    const int i = e * GT + tg, oc = i % OCS, par = i / OCS % PAR, c = i / (OCS * PAR) % 64;
    int n, p;
    row_of(it0 * RPI - 1 + i / (OCS * PAR * 64), n, p);
    before[e] = load_x(n, p, par, c, oc);
  }
  load();
  for (int i = tg; i < RING * S::XV / 16; i += GT) reinterpret_cast<v4u *>(xs)[i] = v4u{0u, 0u, 0u, 0u};
  __syncthreads();   // (the zeros are in place)
#pragma unroll
  for (int e = 0; e < PT; ++e) {
    const int i = e * GT + tg, oc = i % OCS, par = i / OCS % PAR, c = i / (OCS * PAR) % 64, j = i / (OCS * PAR * 64), q = q0 + oc * 8;
    if (j < S::BEFORE) put_x(before[e], keep_first(a.W / ST - q), keep_first((a.W + ST - 1) / ST - q), j, par, c, oc);
  }
  if (ET) {
    for (int i = tg; i < S::BEFORE * PAR * SIDES * 64; i += GT) {
      const int side = i % SIDES, c = i / SIDES & 63, par = i / (SIDES * 64) % PAR, j = i / (SIDES * 64 * PAR);
      int n, p;
      row_of(it0 * RPI - 1 + j, n, p);
      put_edge(load_edge(n, p, par, c, side), j, par, c, side);
    }
  }
  stage(base, 0);
  load();
  __syncthreads();

  const char *const da = dys + half * S::DYO + (wm * 32 + l32) * 16;
  const char *const xb = xs + (wn * 32 + l32) * S::XP * 16 + 12;
  for (int i = 0; i < mine; ++i) {
    const int next_base = slot_of(base, RPI);
    auto prepare = [&]() {   // (the last two iterations stage and request rows that nothing reads)
      stage(next_base, (i + 1) & 1);
      load();
    };
    if (group == 0) prepare();
    if (it0 + i < it1) {
      struct Raw {
        v4u d, e;   // the octet; stride 2: of the even columns
        unsigned l, r;
      };
      const char *const db = da + (i & 1) * S::DYB;
      constexpr int UNITS = OPI / 2 * 3;   // unit u = (step u / 3, row u % 3 of the filter)
      auto read = [&](int u) {
        const int s = u / 3, r = u % 3, oa = 2 * s, ob = 2 * s + 1;
        // the ring row and parity of filter row r under row j of dy
        auto at_of = [&](int o) {
          const int j = o / OCS + (ST == 1 ? r : r == 0 ? 0 : 1);
          return slot_of(base, j) * S::XV + (ST == 2 && r != 1 ? S::XROW : 0) + o % OCS * 16;
        };
        const char *at = OCS % 2 == 0 ? xb + half * 16 + at_of(oa) : xb + (half ? at_of(ob) : at_of(oa));
        Raw w;
        w.l = *reinterpret_cast<const unsigned *>(at);
        w.d = *reinterpret_cast<const v4u *>(at + 4);
        if constexpr (ST == 1) w.r = *reinterpret_cast<const unsigned *>(at + 20);
        else w.e = *reinterpret_cast<const v4u *>(at + 4 + OCS * 16);
        return w;
      };
      struct Taps {
        v4u t[3];
      };
      auto shift = [&](const Raw &w) {
        const unsigned m1 = __builtin_amdgcn_alignbit(w.d[1], w.d[0], 16), m2 = __builtin_amdgcn_alignbit(w.d[2], w.d[1], 16),
                       m3 = __builtin_amdgcn_alignbit(w.d[3], w.d[2], 16);
        Taps o;
        o.t[0] = v4u{__builtin_amdgcn_alignbit(w.d[0], w.l, 16), m1, m2, m3};
        if constexpr (ST == 1) o.t[1] = w.d, o.t[2] = v4u{m1, m2, m3, __builtin_amdgcn_alignbit(w.r, w.d[3], 16)};
        else o.t[1] = w.e, o.t[2] = w.d;
        return o;
      };
      // a unit is read two units ahead and shifted between the matrix instructions of the unit before it
      v4u A[2];
      A[0] = *reinterpret_cast<const v4u *>(db);
      Taps cur = shift(read(0));
      Raw next = read(1);
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        const int s = u / 3, r = u % 3;
        Raw nn = next;
        if (u + 2 < UNITS) nn = read(u + 2);
        if (r == 0 && s + 1 < OPI / 2) A[(s + 1) & 1] = *reinterpret_cast<const v4u *>(db + 2 * (s + 1) * S::DYO);
        const Taps after = shift(next);
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[r * 3 + c] = mfma<BF16>(A[s & 1], cur.t[c], acc[r * 3 + c]);
        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        cur = after, next = nn;
      }
    }
    if (group == 1) prepare();
    base = next_base;
    __syncthreads();
  }

  // ---- sums that are not finite: a zero of the virtual rows and columns may have met an infinity or a NaN.  All of the
  // workgroup's sums are formed again, a row at a time, with every tap's octets in LDS on their own and zero where dy's are no
  // pixels: three to four times the time of the loop above, whatever the values are.  (LDS is free.  Everything is derived anew from opaque
  // copies: what the loop above holds in registers for this, it spills.)
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) bad |= !finite(acc[i][v]);
  int *const again = reinterpret_cast<int *>(smem);
  if (t == 0) *again = 0;
  __syncthreads();
  if (__any(bad) && lane == 0) *again = 1;
  __syncthreads();
  if (*again) {
    static_assert(10 * 64 * OCS * 16 <= S::LDS / 2, "");
    int tt = threadIdx.x, P = a.P, Q = a.Q, H = a.H, W = a.W;
    asm volatile("" : "+v"(tt), "+s"(P), "+s"(Q), "+s"(H), "+s"(W));
    const int th = tt >> 5 & 1, row = wm * 32 + (tt & 31), col = wn * 32 + (tt & 31);
    v4u *const ys = reinterpret_cast<v4u *>(smem + group * (S::LDS / 2)), *const xt = ys + 64 * OCS;   // [channel][octet], [tap][channel][octet]
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
        for (int e = tt & (GT - 1); e < 10 * 64 * OCS; e += GT) {
          const int tap = e / (64 * OCS) - 1, ch = e / OCS % 64, q = q0 + e % OCS * 8;   // tap -1: dy
          const bool of_dy = tap < 0;
          const int h = of_dy ? p : ST * p + tap / 3 - 1, w0 = of_dy ? q : ST * q + tap % 3 - 1, step = of_dy ? 1 : ST;
          const int width = of_dy ? Q : W, height = of_dy ? P : H, channels = of_dy ? a.K : a.C, channel = (of_dy ? k0 : c0) + ch;
          // the first n pixels count, the very first not where it is left of the image: then all come from a column further on
          const int n8 = min(min(8, Q - q), (width - w0 + step - 1) / step), left = w0 < 0, at = w0 + left;
          const bool in = channel < channels && unsigned(h) < unsigned(height);
          const unsigned off = unsigned(((n * channels + channel) * height + h) * width + at) * 2;
          v4u raw[ST];
#pragma unroll
          for (int u = 0; u < ST; ++u)
            raw[u] = of_dy ? load8(rdy, a.dy_bytes, off, in && !u ? width - at : 0) : load8(rx, a.x_bytes, off + 16 * u, in ? width - at - 8 * u : 0);
          v4u o = raw[0];
          if (step == 2) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const v4u &r = raw[ST == 2 ? u / 2 : 0];
              o[u] = __builtin_amdgcn_perm(r[2 * u % 4 + 1], r[2 * u % 4], left ? 0x07060302 : 0x05040100);
            }
          }
          if (left) o = v4u{o[0] << 16, __builtin_amdgcn_alignbit(o[1], o[0], 16), __builtin_amdgcn_alignbit(o[2], o[1], 16),
                            __builtin_amdgcn_alignbit(o[3], o[2], 16)};
          o = in ? o & keep_first(n8) : v4u{0u, 0u, 0u, 0u};
          ys[e] = o;
        }
      }
      __syncthreads();
      if (live && number) {
#pragma unroll 1
        for (int o = 0; o < OCS; o += 2) {
          const bool there = o + th < OCS;
          const int at = there ? o + th : o;
          const v4u d = there ? ys[row * OCS + at] : v4u{0u, 0u, 0u, 0u};
#pragma unroll
          for (int c = 0; c < 9; ++c) {
            const v4u x = xt[(c * 64 + col) * OCS + at];
            acc[c] = mfma<BF16>(d, there ? x : v4u{0u, 0u, 0u, 0u}, acc[c]);
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
  const rsrc_t rp = make_rsrc(a.partial + (size_t(range * a.strips + strip) * a.tiles + tile) * 4 * kAcc, 4 * kAcc * 4);
  const int po = (w4 * kAcc + lane) * 4;
#pragma unroll
  for (int i = 0; i < 9; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, acc[i][v] + ex[(i * 16 + v) * 64]), rp, po, (i * 16 + v) * 256, 0);
}

// dW from the partial images, summed in ascending order.  A workgroup takes four accumulator registers of a wavefront (16 bytes
// a lane) and nine taps: eight filters by 32 channels by nine taps, contiguous stretches of 288 weights; ZL threads share the
// images of a sum, ZL workgroups the taps.
template <int ZL, bool BF16>
__global__ __launch_bounds__(576) void k_wgrad_oct16_reduce(Wo16Args a, int splits, uint16_t *__restrict__ dW) {
  constexpr int TAPS = 9 / ZL;   // taps per workgroup
  typedef float v4f __attribute__((ext_vector_type(4)));
  __shared__ v4f sums[ZL][TAPS][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, z = wave / TAPS, ti = wave % TAPS;
  const int tap0 = int(blockIdx.x) % ZL * TAPS, b = int(blockIdx.x) / ZL, v = b % 4 * 4, w4 = b / 4 % 4, tile = b / 16;
  const size_t image = size_t(a.tiles) * 4 * kAcc;
  const float *p = a.partial + (size_t(tile) * 4 + w4) * kAcc + ((tap0 + ti) * 16 + v) * 64 + lane * 4;
  v4f s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int i = z; i < splits; i += ZL) s += *reinterpret_cast<const v4f *>(p + i * image);
  sums[z][ti][lane] = s;
  __syncthreads();
  for (int e = threadIdx.x; e < TAPS * 256; e += 576) {
    const int l = e / TAPS, tj = e % TAPS;   // l: register, lane of an accumulator
    float r = 0.f;
#pragma unroll
    for (int i = 0; i < ZL; ++i) r += reinterpret_cast<const float *>(sums[i][tj])[l];
    const int k = tile % a.ktiles * 64 + (w4 >> 1) * 32 + 2 * v + 4 * (l >> 5 & 1) + (l >> 6);
    const int c = tile / a.ktiles * 64 + (w4 & 1) * 32 + (l & 31);
    if (k < a.K && c < a.C) dW[(size_t(k) * a.C + c) * 9 + tap0 + tj] = BF16 ? sgh_f32_to_bf16(r) : sgh_f32_to_f16(r);
  }
}

struct Wo16Plan {
  bool ok;
  int ocs, rpi, ktiles, tiles, ranges, strips, iters, per_range;
};

Wo16Plan plan(const sgh_conv_geom *g) {
  Wo16Plan p{};
  if (g->R != 3 || g->S != 3 || g->pad_h != 1 || g->pad_w != 1 || g->stride_h != g->stride_w || g->groups > 1) return p;
  if (g->stride_h != 1 && g->stride_h != 2) return p;
  const size_t lim = size_t(1) << 30;   // byte offsets stay below 2^31
  const size_t xe = size_t(g->N) * g->C * g->H * g->W, ye = size_t(g->N) * g->K * g->P * g->Q;
  // (below 5 G operations no drawn layer gained: the prologue, the exchange and the partial images alone take 20 us)
  if (xe >= lim || ye >= lim || 18.0 * ye * g->C < 5e9) return p;
  const int oc = (g->Q + 7) / 8, st = g->stride_h;
  p.strips = (oc + 3) / 4;
  p.ocs = (oc + p.strips - 1) / p.strips;
  if (st == 2 && p.ocs == 3) p.ocs = 4;   // (two rows of three octets twice over are more than the LDS)
  p.rpi = st == 1 ? (p.ocs == 1 ? 8 : p.ocs == 2 ? 4 : 2) : (p.ocs == 1 ? 4 : p.ocs == 4 ? 1 : 2);
  if (g->P + 1 < p.rpi || size_t(g->N) * (g->P + 1) >= (size_t(1) << 28)) return p;
  p.iters = int((size_t(g->N) * (g->P + 1) + p.rpi - 1) / p.rpi);
  p.ktiles = (g->K + 63) / 64;
  const long tiles = long(p.ktiles) * ((g->C + 63) / 64);
  if (tiles > 16384) return p;
  p.tiles = int(tiles);
  // one workgroup per CU, four iterations each at least; a multiple of eight ranges goes to the XCDs in whole ranges
  long r = sgh_num_cus() / (tiles * p.strips), most = p.iters / 4;
  if (r > most) r = most;
  if (r >= 8) r &= ~7l;
  if (r < 1) r = 1;
  p.per_range = int((p.iters + r - 1) / r);
  p.ranges = r >= 8 ? int(r) : (p.iters + p.per_range - 1) / p.per_range;
  p.ok = true;
  return p;
}

template <int ST, int OCS, int RPI, bool BF16>
int launch(const Wo16Args &a, hipStream_t s) {
  auto kern = k_wgrad_oct16<ST, OCS, RPI, BF16>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) !=
        hipSuccess)
      return SGH_EUNSUPPORTED;
    attr_set = true;
  }
  SGH_LAUNCH_TIMED(kern, dim3(unsigned(a.tiles * a.strips * a.ranges)), dim3(NT), (Shape<ST, OCS, RPI>::LDS + 16), s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

template <bool BF16>
int run(const Wo16Args &a, const Wo16Plan &p, int stride, uint16_t *dW, hipStream_t s) {
  int rc;
  if (stride == 1)
    rc = p.ocs == 4   ? launch<1, 4, 2, BF16>(a, s)
         : p.ocs == 3 ? launch<1, 3, 2, BF16>(a, s)
         : p.ocs == 2 ? launch<1, 2, 4, BF16>(a, s)
                      : launch<1, 1, 8, BF16>(a, s);
  else
    rc = p.ocs == 4   ? launch<2, 4, 1, BF16>(a, s)
         : p.ocs == 2 ? launch<2, 2, 2, BF16>(a, s)
                      : launch<2, 1, 4, BF16>(a, s);
  if (rc != SGH_OK) return rc;
  const int splits = p.ranges * p.strips, blocks = p.tiles * 16;
  if (splits >= 24) hipLaunchKernelGGL((k_wgrad_oct16_reduce<9, BF16>), dim3(blocks * 9), dim3(576), 0, s, a, splits, dW);
  else if (splits >= 6) hipLaunchKernelGGL((k_wgrad_oct16_reduce<3, BF16>), dim3(blocks * 3), dim3(576), 0, s, a, splits, dW);
  else hipLaunchKernelGGL((k_wgrad_oct16_reduce<1, BF16>), dim3(blocks), dim3(576), 0, s, a, splits, dW);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

}  // namespace

size_t sgh_wgrad_oct16_workspace_bytes(const sgh_conv_geom *g) {
  const Wo16Plan p = plan(g);
  return p.ok ? size_t(p.ranges) * p.strips * p.tiles * 4 * kAcc * sizeof(float) : 0;
}

// Fitted as the generic kernel's in conv16.hip: a round's prologue and exchange, the octets that a group walks, partial images
double sgh_wgrad_oct16_us(const sgh_conv_geom *g) {
  const Wo16Plan p = plan(g);
  const double images = double(p.tiles) * p.strips * p.ranges;
  const int rounds = int((p.tiles * long(p.strips) * p.ranges + sgh_num_cus() - 1) / sgh_num_cus());
  const double octets = double(rounds) * ((p.per_range + 1) / 2) * p.ocs * p.rpi;
  return 15 + 29 * (rounds - 1) + octets * (g->stride_h == 1 ? 0.24 : 0.35) + 0.34e-6 * images * 4 * kAcc * sizeof(float);
}

int sgh_wgrad_oct16_run(const sgh_conv_geom *g, const uint16_t *dy, const uint16_t *x, uint16_t *dW, void *workspace, bool bf16,
                        hipStream_t s) {
  const Wo16Plan p = plan(g);
  if (!p.ok) return SGH_EUNSUPPORTED;
  Wo16Args a;
  a.dy = dy, a.x = x, a.partial = static_cast<float *>(workspace);
  a.N = g->N, a.C = g->C, a.K = g->K, a.H = g->H, a.W = g->W, a.P = g->P, a.Q = g->Q;
  a.ktiles = p.ktiles, a.tiles = p.tiles, a.ranges = p.ranges, a.strips = p.strips, a.iters = p.iters, a.per_range = p.per_range;
  a.dy_bytes = unsigned(size_t(g->N) * g->K * g->P * g->Q * 2), a.x_bytes = unsigned(size_t(g->N) * g->C * g->H * g->W * 2);
  sgh_prof_kernel_begin("conv_wgrad16/k_wgrad_oct16", 2.0 * g->N * g->K * g->P * g->Q * double(g->C) * 9);
  const int rc = bf16 ? run<true>(a, p, g->stride_h, dW, s) : run<false>(a, p, g->stride_h, dW, s);
  sgh_prof_kernel_end(s);
  return rc;
}
