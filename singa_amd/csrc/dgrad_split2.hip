// fp32 data gradient of 3x3 convolutions of stride 2 and padding 1 on the bfloat16 matrix instructions, operands split into three
// parts each (conv_split.hip says why that is fp32 arithmetic, and split_parts.h how).
//
//   dx[n][c][h][w] = sum_{k,r,s} dy[n][k][(h + 1 - r) / 2][(w + 1 - s) / 2] * W[k][c][r][s]    where both divide
//
// With (h, w) = (2 p + i, 2 q + j) the nine taps fall into the four classes (i, j): tap (r, s) belongs to i = (r != 1),
// j = (s != 1) and reads dy[p + (r == 0)][q + (s == 0)].  So a workgroup takes BM channels and BN consecutive pixels (p, q) of
// the flattened dy, holds the accumulators of all four classes, and every tap is one product with the slab of dy at an offset of
// its own: no product with the zeros of a dilated gradient, and the 2 x 2 results of a lane's pixel go out in two pieces of 8 bytes.
//
// Each wavefront holds 32 channels x 32 pixels x 4 classes; its six matrix instructions of a tap run while the sum of the tap before goes
// into the accumulators and the operand of the next one comes from LDS.  That takes more than 128 registers, so one workgroup fills
// a CU, and the slab is double-buffered in LDS (one barrier per chunk of 16 channels).  The weights are split and laid out by
// k_conv_split_weights and go from L2 straight to registers, two taps ahead.  A chunk takes 3.1 us, 1.5 of them matrix instructions; what
// the other half waits for are the weights: eight wavefronts fetch 216 KB of fragments per chunk, 30 bytes per clock.  (One tap ahead:
// 3.7; all nine: no better; without the overlap of a tap's sum and the next one's products: 3.3.  64 pixels a wavefront halve the
// fragments, 5.2 us for twice the work, but the tiles are too few and their partial sums too large: 12 per cent faster on 1024 channels and
// 128 images of 28 x 28, 5 to 60 per cent slower on everything below.)
//
// 64 images, whole calls, on fp32 instructions (dgrad3x3.hip) and here: 64 channels of 56 x 56 from 128 100 -> 70 us, 128 of 28 x 28
// from 256 104 -> 64, 256 of 14 x 14 from 512 104 -> 80; 13 images of 40 x 40, 20 x 20 and 10 x 10 36 -> 32, 34 -> 32, 39 -> 34.  Odd
// images ran class by class in igemm.hip: 55 of 38 channels, 16 x 15, from 418 127 -> 34, 45 of 224, 50 x 59, from 213 455 -> 268.  The
// error against float64 is 0.15 to 0.6 times that of those kernels.
//
// Neither the taps of a class nor their signs change within a chunk, so the one that the matrix instructions' rounding needs (it
// leans towards minus infinity) changes from chunk to chunk: in odd ones dy goes negated into the slab and the sums are subtracted.
#include <atomic>
#include <type_traits>

#include "common.h"
#include "dgrad_split2.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

constexpr int NT = 512, NW = NT / 64, KC = 16, TAPS = 9;
constexpr int kOOB = int(0x80000000u);
constexpr int kPos = 48;              // bytes of a slab position: three parts of eight channels
constexpr int kFrag = 3 * 1024;       // bytes of a 32-row weight fragment: three parts x 64 lanes x 16 bytes

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

// The fragments' tap t is the filter's (2 - t / 3, 2 - t % 3)
constexpr int class_of(int t) { return 2 * (t / 3 != 1) + (t % 3 != 1); }
constexpr int down(int t) { return t / 3 == 2; }
constexpr int right(int t) { return t % 3 == 2; }

struct S2Args {
  const float *dy, *W;    // N x K x P x Q, K x C x 3 x 3
  const uint16_t *wt;     // weight fragments [chunk][tap][32-row block][part][lane][8]
  float *dx;              // N x C x H x Wd
  float *partials;        // [workgroup][class][BM][BN]
  int accumulate;         // dx += result
  int N, C, K, P, Q, H, Wd;
  int cblocks, pitch, slab, total_pix, nchunks;
  // Workgroups [0, dp_tiles) take one whole tile each; workgroup dp_tiles + r * share + i takes part i of the chunks of tile
  // dp_tiles + r.
  int ctiles, dp_tiles, share;
  unsigned dy_bytes, wt_bytes, dx_bytes;
};

// The 2 x 2 results of pixel (p, q) for the second pass; `o` is the plane of dx.  Images of odd height or width have no last odd row or
// column.
__device__ __forceinline__ void put(const S2Args &a, float *o, int p, int q, float r00, float r01, float r10, float r11) {
  typedef v2f pair __attribute__((aligned(4)));
  o += size_t(2 * p) * a.Wd + 2 * q;
  const bool below = 2 * p + 1 < a.H;
  if (2 * q + 1 < a.Wd) {
    v2f r0{r00, r01}, r1{r10, r11};
    pair *const o0 = reinterpret_cast<pair *>(o), *const o1 = reinterpret_cast<pair *>(o + a.Wd);
    if (a.accumulate) {
      r0 += *o0;
      if (below) r1 += *o1;
    }
    *o0 = r0;
    if (below) *o1 = r1;
  } else {
    o[0] = a.accumulate ? o[0] + r00 : r00;
    if (below) o[a.Wd] = a.accumulate ? o[a.Wd] + r10 : r10;
  }
}

// GM x (NW / GM) wavefronts, each on 32 channels x 32 pixels of all four classes; ET: slab elements (octet, position) per thread
template <int GM, int ET>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_dgrad_split2(S2Args a) {
  constexpr int GN = NW / GM, BM = GM * 32, BN = GN * 32;
  constexpr int AD = 3;   // weight fragments: this tap's and the next two's
  extern __shared__ __align__(16) char smem[];
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave / GN, wn = wave % GN;
  const int PQ = a.P * a.Q, VH = a.P + 1;     // virtual rows of an image: its own and the zero row below it
  const rsrc_t rdy = make_rsrc(a.dy, a.dy_bytes), rwt = make_rsrc(a.wt, a.wt_bytes);

  const int rest = int(blockIdx.x) - a.dp_tiles, part = rest < 0 ? 0 : rest % a.share;
  const bool whole = rest < 0;
  const int tile = whole ? int(blockIdx.x) : a.dp_tiles + rest / a.share;
  const int ch_begin = whole ? 0 : part * a.nchunks / a.share, ch_end = whole ? a.nchunks : (part + 1) * a.nchunks / a.share;
  const int c0 = (tile % a.ctiles) * BM, pix0 = (tile / a.ctiles) * BN;
  const int n_first = pix0 / PQ, h_first = (pix0 - n_first * PQ) / a.Q;
  const int vbase = n_first * VH + h_first;   // virtual row of the slab's first row

  // ---- slab loader: element e * NT + t = (octet, position); channel k0 + 8 octet + j is the scalar offset j * PQ away
  int g0[ET];
#pragma unroll
  for (int e = 0; e < ET; ++e) {
    const int idx = e * NT + t, oct = idx >= a.slab, pos = idx - (oct ? a.slab : 0);
    const int vr = pos / a.pitch, q = pos - vr * a.pitch, v = vbase + vr, n = v / VH, p = v - n * VH;
    const bool ok = idx < 2 * a.slab && n < a.N && p < a.P && q < a.Q;
    g0[e] = ok ? (((n * a.K + oct * 8) * a.P + p) * a.Q + q) * 4 : kOOB;
  }
  float st[ET][8];
  auto load = [&](int ch, int e, int k_end) {   // (channels from k_end on read as zero)
    const int k0 = ch * KC, valid = k_end - k0 - (e * NT + t >= a.slab ? 8 : 0);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      st[e][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rdy, j < valid ? g0[e] : kOOB, (k0 + j) * PQ * 4, 0));
  };
  const int buffer = 2 * a.slab * kPos;
  auto stage = [&](int e, int to, float sign) {
    v4u p[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Parts s = split2(st[e][2 * i] * sign, st[e][2 * i + 1] * sign);
      p[0][i] = s.p[0], p[1][i] = s.p[1], p[2][i] = s.p[2];
    }
    if (e * NT + t < 2 * a.slab) {
      v4u *d = reinterpret_cast<v4u *>(smem + to + (e * NT + t) * kPos);
      d[0] = p[0], d[1] = p[1], d[2] = p[2];
    }
  };

  // ---- this lane's pixel (column of the B operand)
  auto pixel = [&](int col, int &n, int &p, int &q) {
    const int pix = min(pix0 + col, a.total_pix - 1);   // (a tail lane computes a pixel it does not store)
    n = pix / PQ;
    const int rem = pix - n * PQ;
    p = rem / a.Q, q = rem - p * a.Q;
  };
  int boff;
  {
    int n, p, q;
    pixel(wn * 32 + l32, n, p, q);
    boff = ((n * VH + p - vbase) * a.pitch + q + (lane >> 5) * a.slab) * kPos;
  }

  v16f acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[c][v] = 0.f;

  // ---- weights: step q = chunk * TAPS + tap reads cblocks fragments at q * cblocks * kFrag
  const int step_end = a.nchunks * TAPS, cb = min(c0 / 32 + wm, a.cblocks - 1);   // (rows beyond the last block: computed, not stored)
  v4u wa[AD][3];
  auto weights = [&](v4u (&dst)[3], int step) {
    const int off = (min(step, step_end - 1) * a.cblocks + cb) * kFrag;
#pragma unroll
    for (int p = 0; p < 3; ++p)
      dst[p] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rwt, lane * 16, off + p * 1024, 0));
  };

#pragma unroll
  for (int d = 0; d + 1 < AD; ++d) weights(wa[d], ch_begin * TAPS + d);
  const float first = ch_begin & 1 ? -1.f : 1.f;
#pragma unroll
  for (int e = 0; e < ET; ++e) load(ch_begin, e, a.K);
#pragma unroll
  for (int e = 0; e < ET; ++e) stage(e, 0, first);
  __syncthreads();
  int from = 0;
  v16f sum[2];
#pragma unroll
  for (int v = 0; v < 16; ++v) sum[(TAPS - 1) % 2][v] = 0.f;
  auto accumulate = [&](int tap, float sign) {
    const float f = tap % 2 ? -sign : sign;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[class_of(tap)][v] = __builtin_fmaf(sum[tap % 2][v], f, acc[class_of(tap)][v]);
  };
  for (int ch = ch_begin; ch < ch_end; ++ch) {
    const bool more = ch + 1 < ch_end;
    const float sign = ch & 1 ? -1.f : 1.f;
    const char *const slab = smem + from;
    v4u b[2][3];
    auto fragment = [&](int tap) {
      const char *p = slab + boff + (down(tap) * a.pitch + right(tap)) * kPos;
#pragma unroll
      for (int k = 0; k < 3; ++k) b[tap % 2][k] = *reinterpret_cast<const v4u *>(p + k * 16);
    };
    fragment(0);
    accumulate(TAPS - 1, -sign);   // (of the chunk before; zeros in the first)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tap = 0; tap < TAPS; ++tap) {
      static_assert(TAPS % AD == 0, "ring of the weight fragments");
      const v4u(&w)[3] = wa[tap % AD];
      weights(wa[(tap + AD - 1) % AD], ch * TAPS + tap + AD - 1);
      if (tap < ET) load(ch + 1, tap, more ? a.K : 0);
      if (tap + 1 < TAPS) fragment(tap + 1);
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};   // small products first
#pragma unroll
      for (int v = 0; v < 16; ++v) sum[tap % 2][v] = 0.f;
#pragma unroll
      for (int k = 0; k < 6; ++k) sum[tap % 2] = mfma(w[PA[k]], b[tap % 2][PB[k]], sum[tap % 2]);
      if (tap) accumulate(tap - 1, sign);
      // (into the other buffer, whose readers are behind the last barrier)
      const bool staging = tap >= TAPS - ET;
      if (staging) stage(tap - (TAPS - ET), buffer - from, -sign);
      // (a matrix instruction takes as long as eight others: what there is of these goes between them)
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (staging) __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
        else __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(acc[c]));   // (here, not when the sums of all taps are there)
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    from = buffer - from;
  }
  accumulate(TAPS - 1, (ch_end - 1) & 1 ? -1.f : 1.f);

  bool bad = false;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[c][v] *= kSplitUnscale, bad |= !finite(acc[c][v]);
  // (the slab is free after the last chunk's barrier)
  int *const again = reinterpret_cast<int *>(smem);
  if (t == 0) *again = 0;
  __syncthreads();
  if (__any(bad) && lane == 0) *again = 1;
  __syncthreads();
  if (*again) {
    // What the parts cannot hold (infinities, NaNs, values beyond the scale): the tile from the fp32 values, on the fp32
    // instructions, the slab as [channel][position], the weights from where they are, step k of a tap over channels k and 8 + k.
    // A tap that leaves dy does not exist for that pixel, whatever the weight is: its lanes keep the sum they had.
    float *const xs = reinterpret_cast<float *>(smem);
    int *const numbers = reinterpret_cast<int *>(smem + buffer);   // the last chunk that left a result other than a NaN
    const rsrc_t rw = make_rsrc(a.W, unsigned(size_t(a.K) * a.C * TAPS * 4));
    const int half = lane >> 5, c = min(c0 + wm * 32 + l32, a.C - 1);
    int n, p, q;
    pixel(wn * 32 + l32, n, p, q);
    if (t == 0) *numbers = ch_begin - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
#pragma unroll 1
    for (int ch = ch_begin; ch < ch_end; ++ch) {
#pragma unroll
      for (int e = 0; e < ET; ++e) load(ch, e, a.K);
      float w[2][8];
      auto filter = [&](int tap) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          w[tap % 2][k] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(rw, ch * KC + half * 8 + k < a.K ? ((half * 8 + k) * a.C + c) * TAPS * 4 : kOOB,
                                                          (ch * KC * a.C * TAPS + TAPS - 1 - tap) * 4, 0));
      };
      filter(0);
      __syncthreads();
      if (*numbers < ch - 1) break;
#pragma unroll
      for (int e = 0; e < ET; ++e) {
        const int i = e * NT + t, oct = i >= a.slab;
        if (i < 2 * a.slab)
#pragma unroll
          for (int k = 0; k < 8; ++k) xs[i + (oct * 7 + k) * a.slab] = st[e][k];
      }
      __syncthreads();
#pragma unroll
      for (int tap = 0; tap < TAPS; ++tap) {
        if (tap + 1 < TAPS) filter(tap + 1);
        const float *const xt = xs + boff / kPos + half * 7 * a.slab + down(tap) * a.pitch + right(tap);
        const bool in = (!down(tap) || p + 1 < a.P) && (!right(tap) || q + 1 < a.Q);
        v16f s = acc[class_of(tap)];
#pragma unroll
        for (int k = 0; k < 8; ++k) s = __builtin_amdgcn_mfma_f32_32x32x2f32(w[tap % 2][k], xt[k * a.slab], s, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[class_of(tap)][v] = in ? s[v] : acc[class_of(tap)][v];
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(acc[i]));
      }
      bool any = false;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) any |= acc[i][v] == acc[i][v];
      if (__any(any) && lane == 0) *numbers = ch;
    }
  }

  // ---- store: this lane holds column l32 and rows 8 (v / 4) + 4 (lane / 32) + v % 4 of every 32 x 32 block
  int tt = threadIdx.x;   // (opaque: addresses formed ahead of the matrix instructions would be spilled)
  asm volatile("" : "+v"(tt));
  const int row0 = wm * 32 + (tt >> 3 & 4), col = wn * 32 + (tt & 31);
  if (whole) {
    // A lane's places in the plane of its first channel, those that do not exist out of range; the other channels are scalar offsets away.
    // Results go out in pairs of a row, at any element's address: what a CU's stores cost is their number (rows of an odd number in single
    // floats: 14 filters onto 2 x 360 of 14 x 17 15.0 us, so 9.6, as of 14 x 18).  The last column of such a row goes
    // out with its left neighbour's result, which is the neighbouring lane's and is stored there as well.
    int n, p, q;
    pixel(col, n, p, q);
    const rsrc_t rdx = make_rsrc(a.dx, a.dx_bytes);
    const int plane = a.H * a.Wd * 4, at = int((unsigned(n * a.C + c0 + row0) * a.H * a.Wd + 2 * p * a.Wd + 2 * q) * 4u);
    const bool there = pix0 + col < a.total_pix, below = 2 * p + 1 < a.H, beside = 2 * q + 1 < a.Wd, alone = !beside && (q == 0 || (tt & 31) == 0);
    const int first = there && !alone ? (beside ? at : at - 4) : kOOB, second = there && !alone && below ? first + a.Wd * 4 : kOOB;
    const int left = a.C - c0 - row0;   // channels from this lane's first one on
    auto out = [&](auto acc_c, auto odd_c) {
      constexpr bool ACC = decltype(acc_c)::value, ODD = decltype(odd_c)::value;
#pragma unroll
      for (int v0 = 0; v0 < 16; v0 += 4) {
        if (2 * v0 >= a.C - c0 - wm * 32) break;   // (rows without a channel, of the whole wavefront)
        v2f r[4][2];
        // (the sum in the fixed order result, then what is there; all of it is requested before the first sum is stored)
        if constexpr (ACC)
#pragma unroll
          for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int k = 0; k < 2; ++k)
              r[v][k] = __builtin_bit_cast(
                  v2f, __builtin_amdgcn_raw_buffer_load_b64(rdx, 2 * v0 + v < left ? (k ? second : first) : kOOB, (2 * v0 + v) * plane, 0));
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            v2f w{acc[2 * k][v0 + v], acc[2 * k + 1][v0 + v]};
            if constexpr (ODD) {
              const float own = w[1];   // (a cast of the vector's element itself would take its first)
              constexpr int WAVE_SHR1 = 0x138;
              const float l = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, own), WAVE_SHR1, 0xf, 0xf, true));
              w = beside ? w : v2f{l, w[0]};
            }
            if constexpr (ACC) w += r[v][k];
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, w), rdx, 2 * v0 + v < left ? (k ? second : first) : kOOB,
                                                  (2 * v0 + v) * plane, 0);
          }
      }
      if constexpr (ODD)
        if (__any(alone && there)) {   // (the tile begins with the last column, or it is the only one)
          const int single = alone && there ? at : kOOB, under = alone && there && below ? at + a.Wd * 4 : kOOB;
#pragma unroll
          for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const int rel = 8 * (v >> 2) + (v & 3), off = rel < left ? (k ? under : single) : kOOB;
              float w = acc[2 * k][v];
              if constexpr (ACC) w += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rdx, off, rel * plane, 0));
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w), rdx, off, rel * plane, 0);
            }
        }
    };
    const bool odd = a.Wd & 1;
    if (a.accumulate) odd ? out(std::true_type{}, std::true_type{}) : out(std::true_type{}, std::false_type{});
    else odd ? out(std::false_type{}, std::true_type{}) : out(std::false_type{}, std::false_type{});
    return;
  }
  const rsrc_t rslot = make_rsrc(a.partials + size_t(rest) * (4 * BM * BN), 4 * BM * BN * 4);
  const int off = (row0 * BN + col) * 4;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float r = acc[c][v];
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, r), rslot, off, (c * BM + 8 * (v >> 2) + (v & 3)) * BN * 4, 0);
    }
}

// Sums the parts of the tiles that several workgroups shared, in ascending chunk order: the result does not depend on timing
__global__ __launch_bounds__(256) void k_dgrad_split2_fixup(S2Args a, int BM, int BN) {
  const int r = blockIdx.x, TPR = BN / 4, PQ = a.P * a.Q;
  const int tile = a.dp_tiles + r, c0 = (tile % a.ctiles) * BM, pix0 = (tile / a.ctiles) * BN;
  const int m = int(blockIdx.y * 256 + threadIdx.x) / TPR, col = int(threadIdx.x) % TPR * 4, c = c0 + m;
  if (c >= a.C) return;
  const float *p = a.partials + size_t(r) * a.share * (4 * BM * BN) + m * BN + col;
  v4f s[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) s[k] = *reinterpret_cast<const v4f *>(p + k * BM * BN);
  for (int i = 1; i < a.share; ++i) {
    p += 4 * BM * BN;
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] += *reinterpret_cast<const v4f *>(p + k * BM * BN);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int pix = pix0 + col + j;
    if (pix >= a.total_pix) break;
    const int n = pix / PQ, rem = pix - n * PQ, h = rem / a.Q;
    put(a, a.dx + (size_t(n) * a.C + c) * a.H * a.Wd, h, rem - h * a.Q, s[0][j], s[1][j], s[2][j], s[3][j]);
  }
}

struct S2Plan {
  bool ok;
  int gm, et, bm, bn, pitch, slab, nchunks, cblocks;
  int ctiles, tiles, dp_tiles, share, wgs;
};

S2Plan plan(const sgh_conv_geom *g) {
  S2Plan p{};
  if (g->R != 3 || g->S != 3 || g->stride_h != 2 || g->stride_w != 2 || g->pad_h != 1 || g->pad_w != 1) return p;
  if (g->P != (g->H + 1) / 2 || g->Q != (g->W + 1) / 2) return p;
  if (g->K < 8) return p;   // (see conv_split.hip)
  const size_t lim = size_t(1) << 31;
  if (size_t(g->N) * g->K * g->P * g->Q * 4 >= lim || size_t(g->N) * g->C * g->H * g->W * 4 >= lim) return p;
  if (size_t(g->N) * (g->P + 1) >= lim / 64) return p;
  p.pitch = g->Q + 1;
  p.nchunks = (g->K + KC - 1) / KC;
  p.cblocks = (g->C + 31) / 32;
  if (size_t(p.nchunks) * TAPS * p.cblocks * kFrag >= lim) return p;
  // Tile: 128 channels x 64 pixels, or 64 x 128 where that leaves fewer rows without a channel (128 channels of 28 x 28 64 / 68 us; 133
  // channels of 38 x 34 37 / 32).
  const int pq = g->P * g->Q, r128 = (g->C + 127) / 128 * 128, r64 = (g->C + 63) / 64 * 64;
  p.gm = r128 == r64 ? 4 : 2;
  p.bm = p.gm * 32, p.bn = NW / p.gm * 32;
  // virtual rows a tile can touch: its pixel rows, the row below, and the zero row of every image boundary it crosses
  p.slab = ((p.bn + g->Q - 2) / g->Q + 2 + (p.bn - 1) / pq + 1) * p.pitch;
  p.et = 2 * p.slab <= 2 * NT ? 2 : 3;
  if (2 * p.slab > 3 * NT) return p;
  // Whole multiples of the CU count of tiles are one workgroup's each; the chunks of a remaining tile are dealt evenly to as many
  // workgroups as leave every CU at most one of them.
  const int cus = sgh_num_cus();
  p.ctiles = (g->C + p.bm - 1) / p.bm;
  const long tiles = long(p.ctiles) * ((long(g->N) * pq + p.bn - 1) / p.bn);
  if (tiles >= (long(1) << 30)) return p;
  // (two or three chunks, few tiles: their sums cost what the split saves.  31 channels onto 5 x 131 of 9 x 11 15.6 us on fp32
  // instructions, 18.0 here; 38 onto 2 x 407 of 8 x 9 17.9 / 18.5; 35 onto 3 x 506 of 46 x 62, 136 tiles, 40 / 23)
  if ((p.nchunks == 2 || p.nchunks == 3) && 2 * tiles < cus) return p;
  p.tiles = int(tiles);
  p.dp_tiles = int(tiles / cus * cus);
  const int rest = p.tiles - p.dp_tiles;
  p.share = rest ? cus / rest : 1;
  if (p.share > p.nchunks) p.share = p.nchunks;
  if (p.share <= 1) p.share = 1, p.dp_tiles = p.tiles;
  p.wgs = p.dp_tiles + (p.tiles - p.dp_tiles) * p.share;
  p.ok = true;
  return p;
}

template <int GM, int ET>
int launch(const S2Args &a, const S2Plan &p, hipStream_t s) {
  auto kern = k_dgrad_split2<GM, ET>;
  static std::atomic<bool> allowed{false};   // (host threads may come here at once)
  if (!allowed.load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
      return SGH_EUNSUPPORTED;
    allowed.store(true, std::memory_order_relaxed);
  }
  SGH_LAUNCH_TIMED(kern, dim3(unsigned(p.wgs)), dim3(NT), size_t(p.slab) * 4 * kPos, s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

inline size_t align256(size_t v) { return (v + 255) & ~size_t(255); }
inline size_t weight_bytes(const S2Plan &p) { return size_t(p.nchunks) * TAPS * p.cblocks * kFrag; }

}  // namespace

bool sgh_dgrad_split2_supported(const sgh_conv_geom *g) { return !sgh_env().conv_split_off && plan(g).ok; }

size_t sgh_dgrad_split2_workspace_bytes(const sgh_conv_geom *g) {
  const S2Plan p = plan(g);
  return p.ok ? align256(weight_bytes(p)) + size_t(p.wgs - p.dp_tiles) * 4 * p.bm * p.bn * sizeof(float) : 0;
}

int sgh_dgrad_split2_run(const sgh_conv_geom *g, const float *dy, const float *W, float *dx, void *workspace, hipStream_t s,
                         bool accumulate) {
  const S2Plan p = plan(g);
  if (!p.ok) return SGH_EUNSUPPORTED;
  S2Args a;
  a.dy = dy, a.W = W, a.dx = dx;
  a.wt = static_cast<const uint16_t *>(workspace);
  a.partials = reinterpret_cast<float *>(static_cast<char *>(workspace) + align256(weight_bytes(p)));
  a.accumulate = accumulate ? 1 : 0;
  a.N = g->N, a.C = g->C, a.K = g->K, a.P = g->P, a.Q = g->Q, a.H = g->H, a.Wd = g->W;
  a.cblocks = p.cblocks, a.pitch = p.pitch, a.slab = p.slab, a.total_pix = g->N * g->P * g->Q, a.nchunks = p.nchunks;
  a.ctiles = p.ctiles, a.dp_tiles = p.dp_tiles, a.share = p.share;
  a.dy_bytes = unsigned(size_t(g->N) * g->K * g->P * g->Q * 4), a.wt_bytes = unsigned(weight_bytes(p));
  a.dx_bytes = unsigned(size_t(g->N) * g->C * g->H * g->W * 4);
  int rc = SGH_EUNSUPPORTED;
  sgh_prof_kernel_begin("conv_dgrad/k_dgrad_split2", 2.0 * g->N * g->K * g->P * g->Q * g->C * TAPS);
#define S2_CASE(GM_, ET_) \
  if (p.gm == GM_ && p.et == ET_) rc = launch<GM_, ET_>(a, p, s);
  S2_CASE(4, 2) S2_CASE(4, 3) S2_CASE(2, 2) S2_CASE(2, 3)
#undef S2_CASE
  sgh_prof_kernel_end(s);
  if (rc != SGH_OK) return rc;
  if (p.share > 1) {
    hipLaunchKernelGGL(k_dgrad_split2_fixup, dim3(unsigned(p.tiles - p.dp_tiles), unsigned(p.bm * p.bn / 1024)), dim3(256), 0, s, a, p.bm,
                       p.bn);
    if (hipGetLastError() != hipSuccess) return SGH_EINVAL;
  }
  return SGH_OK;
}
