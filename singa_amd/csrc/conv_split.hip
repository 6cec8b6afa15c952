// fp32 convolutions of stride 1 with "same" padding (3x3, 5x5), forward and data gradient, and 3x3 forward passes of stride 2, on the
// bfloat16 matrix instructions without giving up fp32 operands (the splitting of G. Henry, P. Tang, A. Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", 2019): a fp32 value, times 2^16 so that this holds for
// the smallest ones too, is the sum of three bfloat16 values
//
//   x = x0 + x1 + x2,   x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1)      (8 + 8 + 8 bits of significand)
//
// and a product of two of them is the sum of nine exact products, of which the six with weights down to 2^-16 are formed
// (x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0).  The three left out come to 2^-24 of the product at most, 2^-28 in the mean.
// v_mfma_f32_32x32x16_bf16 multiplies 16 x as much per cycle as v_mfma_f32_32x32x2_f32, so six of them are 2.67 times as
// fast, with fp32 accumulators either way.
//
// What decides the error of a convolution is how often its sum is rounded: the fp32 instructions do that once per product, the
// bfloat16 ones once per eight, six times over.  So the six products of a tap and 16 channels are summed on their own, the
// small ones first, and that sum is added to the accumulator with one rounding to nearest.  (All on the accumulator: 1.05 to 1.2
// times the error of the fp32 instructions behind a ReLU, whose zeros cost those nothing.)  The matrix instructions round towards
// minus infinity on average; the weights of every other tap are negated, and their sums subtracted, so that this does not add
// up (900 channels: a mean error of 2e-7 of the results with one sign, 2e-8 with two).
//
//   out[n][c][h][w] = sum_{k,r,s} in[n][k][h + r - o][w + s - o] * Wf[c][k][r][s],   o = (R - 1) / 2
//
// (forward passes of 3x3 and stride 2 as well: in[n][k][2 h + r - o][2 w + s - o])
//
// forward: Wf = W; data gradient: Wf[c][k][r][s] = W[k][c][R - 1 - r][R - 1 - s].
//
// GEMM view: M = output channels, N = consecutive pixels of the flattened (n, h, w) index, reduction = (k, tap) in chunks of
// 16 input channels.  Per chunk a workgroup stages the input rows its pixels touch, split, as [octet of channels][slab
// position][part][8 channels]: 48 bytes per position, one operand fragment of a tap is three ds_read_b128 at an offset that
// is the tap's alone.  A value is fetched and split once per chunk for all R * R taps.  Rows are addressed in a "virtual row"
// space in which every image owns P + 2 o rows, so a tile may straddle images and the padding is materialised as zeros.
// The weights are split and laid out in fragment order by a kernel of their own and go from L2 straight to registers, a tap or two
// ahead: no LDS, no barrier per tap.
//
// 512 threads = 8 wavefronts of at most 128 registers, two workgroups per CU where the slab takes no more than 80 KB of LDS: while
// one stages and waits at its barriers the other one's matrix instructions run.
//
// Stride 2, whole forward calls, the generic kernel (igemm.hip) and here: 64 images of 64 channels, 56 x 56, to 128 125 -> 99 us, of 128,
// 28 x 28, to 256 163 -> 69, of 256, 14 x 14, to 512 169 -> 77; 13 of 256, 10 x 10, to 512 108 -> 33 (48 workgroups before); the error
// 0.12 to 0.35 times, and over 34 drawn layers none slower than 0.97.  The tiles are the ones of stride 1; a wavefront of two blocks with
// three slab elements a thread, ten registers spilled, is faster than one block (28 x 28: 69 / 75, 14 x 14: 77 / 92).
//
// 64 images, whole calls, on fp32 instructions (dgrad3x3.hip) and here: 64 channels of 56 x 56 forward 143 -> 97 us, data gradient
// 131 -> 90; 128 of 28 x 28 139 -> 94, 128 -> 90; 256 of 14 x 14 145 -> 97, 136 -> 91; 512 of 7 x 7 156 -> 106, 137 -> 100.  The error
// against float64 is 0.15 to 0.6 times that of the fp32 instructions, 0.9 at most, on normal, on rectified and on positive
// operands; an addition of 16 results per six products costs 4 to 8 per cent of the time.
//
// Infinities, NaNs and values and results too large for the scale (2^112, 2^96): parts that overflow make NaNs, so a tile with a result that comes out non-finite is formed again by its workgroup on the fp32 matrix
// instructions, whatever the values are.
#include "common.h"
#include "conv_split.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int NT = 512, NW = NT / 64, KC = 16;
constexpr int kOOB = int(0x80000000u);
constexpr int kMaxSlab = 1024;        // positions of a slab (96 KB; up to 853 of them leave room for a second workgroup)
constexpr int kPos = 48;              // bytes of a slab position: three parts of eight channels
constexpr int kFrag = 3 * 1024;       // bytes of a 32-row weight fragment: three parts x 64 lanes x 16 bytes

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

// Eight fp32 values -> the three parts of each, packed
__device__ __forceinline__ void split8(const float (&v)[8], v4u (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const Parts s = split2(v[2 * i], v[2 * i + 1]);
    part[0][i] = s.p[0], part[1][i] = s.p[1], part[2][i] = s.p[2];
  }
}

struct ScArgs {
  const float *in;
  const float *W;         // the weights, W[c * w_c + k * w_k + tap]; the data gradient takes the taps in reverse
  int w_c, w_k;
  const uint16_t *wt;     // weight fragments [chunk][tap][32-row block][part][lane][8]
  const float *bias;      // per output channel (NULL: none)
  float *out;
  float *partials;        // [workgroup][BM * BN]
  int accumulate;         // out += result
  int dgrad;
  int N, C, K, P, Q;      // in is N x K x IH x IW, out N x C x P x Q
  int IH, IW, plane;      // P and Q at stride 1; bytes of IH x IW
  int cblocks;            // 32-row blocks of the weight fragments
  int pitch, slab;        // LDS row pitch and positions of the slab (rows * pitch)
  int total_pix, nchunks;
  // Workgroups [0, dp_tiles) take one whole tile each; workgroup dp_tiles + r * share + i takes part i of the chunks of tile
  // dp_tiles + r.  Its slot of `partials` holds what it leaves for k_conv_split_fixup.
  int ctiles, dp_tiles, share;
  int xcd_runs;
  unsigned in_bytes, wt_bytes;
};

__device__ __forceinline__ int whole_tile_of(const ScArgs &a, int w) {   // see dgrad3x3.hip: runs of eight tiles per XCD
  if (!a.xcd_runs) return w;
  const int x = w & 7, j = w >> 3;
  return (((j >> 3) << 3) + x) * 8 + (j & 7);
}

// Column of the input at place `at` of a slab row, from the left padding on, and the other way round.  At stride 2 the even columns come
// first, then the odd ones, so that neighbouring pixels read neighbouring places for every tap.
template <int ST>
__device__ __forceinline__ int column_at(int at, int pitch) {
  const int even = (pitch + 1) >> 1;
  return ST == 1 ? at : at < even ? 2 * at : 2 * (at - even) + 1;
}
template <int ST>
__device__ __forceinline__ int place_of(int column, int pitch) {
  return ST == 1 ? column : (column & 1) * ((pitch + 1) >> 1) + (column >> 1);
}

// GM x (NW / GM) wavefronts, each on WM x WN blocks of 32 x 32; ET: slab elements (octet, position) per thread; R: filter size;
// ST: stride (2: forward passes only).
template <int GM, int WM, int WN, int ET, int R, int ST>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_conv_split(ScArgs a) {
  constexpr int GN = NW / GM, BM = GM * WM * 32, BN = GN * WN * 32, TAPS = R * R, O = (R - 1) / 2;
  // Weight fragments: this tap's and the next one's, or the next two's where a wavefront has six products per tap and not twelve to cover
  // the loads (5x5 onto 64 channels, 128 images of 16 x 16: 29.3 -> 26.8 us, onto 32 35.2 -> 33.4; 64 channels, 8 x 56 x 56: 25.4 -> 23.6)
  constexpr int AD = WN == 1 ? 3 : 2;
  constexpr int EARLY = WN > 1 && ET > 3 ? 3 : ET;   // elements requested under the products (registers); the others after them
  extern __shared__ __align__(16) char smem[];
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave / GN, wn = wave % GN;
  const int PQ = a.P * a.Q, IH = ST == 1 ? a.P : a.IH, IW = ST == 1 ? a.Q : a.IW, VH = IH + 2 * O;
  const rsrc_t rin = make_rsrc(a.in, a.in_bytes), rwt = make_rsrc(a.wt, a.wt_bytes);

  const int rest = int(blockIdx.x) - a.dp_tiles, part = rest < 0 ? 0 : rest % a.share;
  const bool whole = rest < 0;
  const int tile = whole ? whole_tile_of(a, int(blockIdx.x)) : a.dp_tiles + rest / a.share;
  const int ch_begin = whole ? 0 : part * a.nchunks / a.share, ch_end = whole ? a.nchunks : (part + 1) * a.nchunks / a.share;
  const int c0 = (tile % a.ctiles) * BM, pix0 = (tile / a.ctiles) * BN;
  const int n_first = pix0 / PQ, h_first = (pix0 - n_first * PQ) / a.Q;
  const int vbase = n_first * VH + h_first * ST;   // virtual row of the slab's first row

  // ---- slab loader: element e * NT + t = (octet, position); channel k0 + 8 octet + j is the scalar offset j * IH * IW away
  int g0[ET];
#pragma unroll
  for (int e = 0; e < ET; ++e) {
    const int idx = e * NT + t, oct = idx >= a.slab, pos = idx - (oct ? a.slab : 0);
    const int vr = pos / a.pitch, col = column_at<ST>(pos - vr * a.pitch, a.pitch), v = vbase + vr, n = v / VH;
    const int p = v - n * VH - O, q = col - O;
    const bool ok = idx < 2 * a.slab && n < a.N && unsigned(p) < unsigned(IH) && unsigned(q) < unsigned(IW);
    g0[e] = ok ? (((n * a.K + oct * 8) * IH + p) * IW + q) * 4 : kOOB;
  }
  float st[ET][8];
  // (no branch: behind one, the waits for the weights would have to count on none of these loads and wait for them too.
  // Channels from `k_end` on read as zero: those beyond K, and all of them when there is no further chunk.)
  auto load = [&](int ch, int e, int k_end) {
    const int k0 = ch * KC, valid = k_end - k0 - (e * NT + t >= a.slab ? 8 : 0);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      st[e][j] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rin, j < valid ? g0[e] : kOOB, ST == 1 ? (k0 + j) * PQ * 4 : (k0 + j) * a.plane, 0));
  };
  auto stage = [&]() {
#pragma unroll
    for (int e = 0; e < ET; ++e) {
      v4u part[3];
      split8(st[e], part);
      if (e * NT + t < 2 * a.slab) {
        v4u *d = reinterpret_cast<v4u *>(smem + (e * NT + t) * kPos);
        d[0] = part[0], d[1] = part[1], d[2] = part[2];
      }
    }
  };

  // ---- this lane's pixels (columns of the B operand)
  int boff[WN], pixn[WN];
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int pix = min(pix0 + (wn * WN + j) * 32 + l32, a.total_pix - 1);   // (a tail lane computes a pixel it does not store)
    const int pn = pix / PQ, prem = pix - pn * PQ, ph = prem / a.Q, pw = prem - ph * a.Q;
    boff[j] = ((pn * VH + ph * ST - vbase) * a.pitch + pw + (lane >> 5) * a.slab) * kPos;   // (place_of an even column: pw)
    pixn[j] = pn;
  }

  v16f acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // ---- weights: step q = chunk * TAPS + tap reads cblocks fragments at q * cblocks * kFrag, `step_end` steps in all
  const int step_end = a.nchunks * TAPS, cb = c0 / 32 + wm * WM;
  v4u wa[AD][WM][3];
  auto weights = [&](v4u (&dst)[WM][3], int step) {
    const int base = min(step, step_end - 1) * a.cblocks;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int off = (base + min(cb + i, a.cblocks - 1)) * kFrag;   // (rows beyond the last block: computed, not stored)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        dst[i][p] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rwt, lane * 16, off + p * 1024, 0));
    }
  };

  // operand fragment of block j at a tap
  v4u b[3];
  auto fragment = [&](int tap, int j) {
    const char *p = smem + boff[j] + (tap / R * a.pitch + place_of<ST>(tap % R, a.pitch)) * kPos;
#pragma unroll
    for (int k = 0; k < 3; ++k) b[k] = *reinterpret_cast<const v4u *>(p + k * 16);
  };

  // Everything a tap needs is requested before the matrix instructions of an earlier one: weights AD - 1 taps ahead, the next
  // chunk's slab an element per tap, a block's fragment while the other block is multiplied.  (The scheduling barriers keep
  // the compiler from moving the requests down to their uses, which it does to save registers.)
#pragma unroll
  for (int e = 0; e < ET; ++e) load(ch_begin, e, a.K);
  weights(wa[0], ch_begin * TAPS);
  if (AD > 2) weights(wa[1], ch_begin * TAPS + 1);
  stage();
  __syncthreads();
  const rsrc_t rslot = make_rsrc(a.partials + size_t(whole ? 0 : rest) * (BM * BN), BM * BN * 4);
  const int slot_off = ((wm * WM * 32 + 4 * (lane >> 5)) * BN + wn * WN * 32 + l32) * 4;
  auto keep = [&](float r, int off, int row) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, r), rslot, off, row, 0);
  };
  auto slot_row = [](int i, int j, int v) { return ((i * 32 + 8 * (v >> 2) + (v & 3)) * BN + j * 32) * 4; };   // (scalar)
  for (int ch = ch_begin; ch < ch_end; ++ch) {
    const bool more = ch + 1 < ch_end;
    fragment(0, 0);
#pragma unroll
    for (int tap = 0; tap < TAPS; ++tap) {
      const v4u(&w)[WM][3] = wa[tap % AD];
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        if (j == 0) weights(wa[(tap + AD - 1) % AD], ch * TAPS + tap + AD - 1);
        if (j == WN - 1 && tap < EARLY) load(ch + 1, tap, more ? a.K : 0);
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};   // small products first
        v16f sum[WM];
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) sum[i][v] = 0.f;
#pragma unroll
        for (int k = 0; k < 6; ++k)
#pragma unroll
          for (int i = 0; i < WM; ++i) sum[i] = mfma(w[i][PA[k]], b[PB[k]], sum[i]);
        __builtin_amdgcn_sched_barrier(0);
        if (j + 1 < WN) fragment(tap, j + 1);
        else if (tap + 1 < TAPS) fragment(tap + 1, 0);
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          acc[i][j] = tap % 2 ? acc[i][j] - sum[i] : acc[i][j] + sum[i];
          asm volatile("" : "+v"(acc[i][j]));   // (here, not when all taps' sums are there)
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int e = EARLY; e < ET; ++e) load(ch + 1, e, more ? a.K : 0);
    if (TAPS % AD) {   // (the ring continues one place further)
      static_assert(TAPS % AD == 0 || TAPS % AD == 1, "ring of the weight fragments");
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const v4u x = wa[0][i][p];
#pragma unroll
          for (int d = 0; d + 1 < AD; ++d) wa[d][i][p] = wa[d + 1][i][p];
          wa[AD - 1][i][p] = x;
        }
    }
    __syncthreads();
    if (more) {
      stage();
      __syncthreads();
    }
  }

  // ---- store: this lane holds column l32 and rows 8 (v / 4) + 4 (lane / 32) + v % 4 of every 32 x 32 block
  const int lhalf = lane >> 5;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] *= kSplitUnscale, bad |= !finite(acc[i][j][v]);
  auto put = [&](int m, int col, int n, float r) {   // row, column of the tile
    const int c = c0 + m, pix = pix0 + col;
    if (c >= a.C || pix >= a.total_pix) return;
    float *o = a.out + (size_t(n) * a.C + c) * PQ + (pix - n * PQ);
    if (a.bias) r += a.bias[c];
    *o = a.accumulate ? *o + r : r;
  };
  // (the slab is free after the last chunk's barrier)
  int *const again = reinterpret_cast<int *>(smem);
  if (t == 0) *again = 0;
  __syncthreads();
  if (__any(bad) && lane == 0) *again = 1;
  __syncthreads();
  if (*again) {
    // The tile from the fp32 values, on the fp32 instructions: the slab as [channel][position], the weights from where they are,
    // step k of a tap over channels k and 8 + k.  Taps in the padding multiply a zero in the forward pass (which makes a NaN of an
    // infinite weight) and do not exist in the data gradient, where an infinite or NaN weight is multiplied pixel by pixel.
    // (Everything is derived anew from opaque copies: what the loop above holds in registers for this, it spills.)
    static_assert(WM == 1, "");
    float *const xs = reinterpret_cast<float *>(smem);
    int tt = threadIdx.x, P = IH, Q = IW, slab = a.slab, pitch = a.pitch;   // (of the input)
    asm volatile("" : "+v"(tt), "+s"(P), "+s"(Q), "+s"(slab), "+s"(pitch));
    const int half = tt >> 5 & 1, column = tt & 31, c = min(c0 + wm * 32 + column, a.C - 1), vh = P + 2 * O;
    int ph[WN], pw[WN], base[WN];   // this lane's pixels: row, column, place in the slab of channel 8 half
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int pix = min(pix0 + (wn * WN + j) * 32 + column, a.total_pix - 1), pq = ST == 1 ? P * Q : PQ, qq = ST == 1 ? Q : a.Q, n = pix / pq, rem = pix - n * pq;
      ph[j] = rem / qq, pw[j] = rem - ph[j] * qq;
      base[j] = (n * vh + ph[j] * ST - vbase) * pitch + pw[j] + half * 8 * slab;
    }
    // not every result of this wavefront, of the workgroup is a NaN yet (in a diverged network they soon are)
    bool number = true;
    int *const numbers = reinterpret_cast<int *>(smem + 2 * a.slab * kPos);   // the last chunk that left one
    if (tt == 0) *numbers = ch_begin - 1;
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[0][j][v] = 0.f;
    for (int ch = ch_begin; ch < ch_end; ++ch) {
      __syncthreads();
      if (*numbers < ch - 1) break;
#pragma unroll 1
      for (int i = tt; i < 2 * slab; i += NT) {
        const int oct = i >= slab, pos = i - (oct ? slab : 0), vr = pos / pitch, q = column_at<ST>(pos - vr * pitch, pitch) - O, v = vbase + vr, n = v / vh;
        const int p = v - n * vh - O, k0 = ch * KC + oct * 8;
        const bool in = n < a.N && unsigned(p) < unsigned(P) && unsigned(q) < unsigned(Q);
        const float *const src = a.in + ((size_t(n) * a.K + k0) * P + p) * Q + q;
#pragma unroll
        for (int k = 0; k < 8; ++k) xs[(oct * 8 + k) * slab + pos] = in && k0 + k < a.K ? src[size_t(k) * P * Q] : 0.f;
      }
      __syncthreads();
#pragma unroll 1
      for (int i = 0; i < TAPS && number; ++i) {
        // (the middle tap first: it is inside the image everywhere, so a layer of NaN weights ends here)
        const int tap = (i + TAPS / 2) % TAPS;
        const bool apart = a.dgrad && i;
        const float *const wp = a.W + size_t(c) * a.w_c + (a.dgrad ? TAPS - 1 - tap : tap);
        const int k0 = ch * KC + half * 8;
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = k0 + k < a.K ? wp[size_t(k0 + k) * a.w_k] : 0.f;
        const float *const xt = xs + tap / R * pitch + place_of<ST>(tap % R, pitch);
        if (apart) {
#pragma unroll 1
          for (int k = 0; k < 8; ++k) {
            float wk = w[0];
#pragma unroll
            for (int u = 1; u < 8; ++u) wk = k == u ? w[u] : wk;
            for (unsigned long long m = __ballot(!finite(wk)); m; m &= m - 1) {
              const int from = __builtin_ctzll(m), row = from & 31;
              const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wk), from));
#pragma unroll
              for (int j = 0; j < WN; ++j) {
                const bool in = unsigned(ph[j] + tap / R - O) < unsigned(P) && unsigned(pw[j] + tap % R - O) < unsigned(Q);
                const float x = xt[base[j] + ((from >> 5) - half) * 8 * slab + k * slab];
#pragma unroll
                for (int v = 0; v < 16; ++v)
                  if (v == (row >> 3) * 4 + (row & 3) && in && half == (row >> 2 & 1)) acc[0][j][v] = __builtin_fmaf(f, x, acc[0][j][v]);
              }
            }
          }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float f = apart && !finite(w[k]) ? 0.f : w[k];
#pragma unroll
          for (int j = 0; j < WN; ++j)
            acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f, xt[base[j] + k * slab], acc[0][j], 0, 0, 0);
        }
        bool any = false;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) any |= acc[0][j][v] == acc[0][j][v];
        number = __any(any);
      }
      if (number && lane == 0) *numbers = ch;
    }
  }
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = (wm * WM + i) * 32 + 8 * (v >> 2) + 4 * lhalf + (v & 3), col = (wn * WN + j) * 32 + l32;
        if (whole) put(m, col, pixn[j], acc[i][j][v]);
        else keep(acc[i][j][v], slot_off, slot_row(i, j, v));
      }
}

// Sums the parts of the tiles that several workgroups shared, in ascending chunk order: the result does not depend on timing
__global__ __launch_bounds__(256) void k_conv_split_fixup(ScArgs a, int BM, int BN) {
  const int r = blockIdx.x, TPR = BN / 4;
  const int tile = a.dp_tiles + r, c0 = (tile % a.ctiles) * BM, pix0 = (tile / a.ctiles) * BN, PQ = a.P * a.Q;
  const int m = int(blockIdx.y * 256 + threadIdx.x) / TPR, col = int(threadIdx.x) % TPR * 4, c = c0 + m;
  if (c >= a.C) return;
  const float *p = a.partials + size_t(r) * a.share * BM * BN + m * BN + col;
  v4f s = *reinterpret_cast<const v4f *>(p);
  for (int i = 1; i < a.share; ++i) s += *reinterpret_cast<const v4f *>(p + size_t(i) * BM * BN);
  const float bb = a.bias ? a.bias[c] : 0.f;
  int pix = pix0 + col, pn = pix / PQ, prem = pix - pn * PQ;
  if ((PQ & 3) == 0 && pix + 3 < a.total_pix) {   // the four pixels lie in one image, 16-byte aligned
    v4f *o = reinterpret_cast<v4f *>(a.out + (size_t(pn) * a.C + c) * PQ + prem);
    *o = a.accumulate ? *o + (s + bb) : s + bb;
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j, ++pix) {
    if (pix >= a.total_pix) break;
    float *o = a.out + (size_t(pn) * a.C + c) * PQ + prem;
    *o = a.accumulate ? *o + (s[j] + bb) : s[j] + bb;
    if (++prem == PQ) prem = 0, ++pn;
  }
}

inline size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

}  // namespace

sgh_conv_split_plan sgh_conv_split_plan_of(const sgh_conv_geom *g) {
  sgh_conv_split_plan p{};
  if (sgh_env().conv_split_off) return p;
  // (stride 2: the geometry of a forward pass with its channels swapped)
  if ((g->R != 3 && g->R != 5) || g->S != g->R || g->stride_h != g->stride_w || g->stride_h < 1 || g->stride_h > (g->R == 3 ? 2 : 1)) return p;
  const int o = (g->R - 1) / 2;
  p.st = g->stride_h, p.ih = p.st == 1 ? g->P : g->H, p.iw = p.st == 1 ? g->Q : g->W;
  if (g->pad_h != o || g->pad_w != o) return p;
  // (below eight channels the padded reduction rounds more often than the fp32 instructions do on the few products there are:
  // 5x5 over 3 channels 1.5e-7 -> 2.0e-7 from float64)
  if (g->K < 8) return p;
  const size_t lim = size_t(1) << 31;
  if (size_t(g->N) * g->K * p.ih * p.iw * 4 >= lim || size_t(g->N) * g->C * g->P * g->Q * 4 >= lim) return p;
  if (size_t(g->N) * (p.ih + 2 * o) >= lim / 64) return p;
  p.r = g->R;
  p.pitch = (g->Q - 1) * p.st + p.r;
  p.nchunks = (g->K + KC - 1) / KC;
  p.cblocks = (g->C + 31) / 32;
  if (size_t(p.nchunks) * p.r * p.r * p.cblocks * kFrag >= lim) return p;
  const int cus = sgh_num_cus();
  const long pixels = long(g->N) * g->P * g->Q;
  // Tile: 128 x 128, 64 x 256, 64 x 128 or 32 x 256 (a wavefront holds 32 x 64 of the first two, 32 x 32 of the others), the
  // least rows counting those beyond C, with 32-row tiles a quarter dearer.  64 rows take 256 pixels from two fifths more
  // tiles than CUs on; below, tiles of half the size leave fewer CUs idle (64 channels of 56 x 56: N = 64 94 against 105 us,
  // N = 32 58 against 57, N = 8 32 against 29; 96 channels of 20 x 20: 51 on 32 rows, 57 on 128; 200 channels: 42 on 128, 54 on 32).
  auto rows_of = [&](int bm) { return (g->C + bm - 1) / bm * bm; };
  const int r128 = rows_of(128), r64 = rows_of(64), r32 = rows_of(32);
  auto take = [&](int gm, int wn) {
    p.gm = gm, p.wm = 1, p.wn = wn, p.bm = gm * 32, p.bn = NW / gm * wn * 32;
    // virtual rows a tile can touch: its pixel rows, the halo rows, and the zero rows of every image boundary it crosses
    const int vh = p.ih + 2 * o, pq = g->P * g->Q;
    p.rows = (p.bn + g->Q - 2) / g->Q * p.st + p.r + (vh - g->P * p.st) * ((p.bn - 1) / pq + 1);
    int a = pq, b = p.bn;   // the distinct places in an image where a tile begins, if they are few: not the bound but what it is
    while (b) {
      const int m = a % b;
      a = b, b = m;
    }
    if (p.st > 1 && pq / a <= 256) {
      p.rows = 0;
      for (int first = 0; first < pq; first += a) {
        const int last = first + p.bn - 1;
        const int rows = last / pq * vh + last % pq / g->Q * p.st + p.r - first / g->Q * p.st;
        if (rows > p.rows) p.rows = rows;
      }
    }
    return long(p.rows) * p.pitch <= (p.st > 1 && wn > 1 ? 3 * NT / 2 : kMaxSlab);   // (four elements per thread: spills)
  };
  bool fits = false;
  // (too few chunks to give every CU one: small tiles.  204 filters over 14 channels, 10 x 2 tiles: 16.5 -> 13 us)
  if (p.r == 3 && r128 == r64 && 4 * r128 <= 5 * r32 && r128 / 128 * ((pixels + 127) / 128) * p.nchunks >= cus) fits = take(4, 2);
  if (!fits && 4 * r64 <= 5 * r32)
    fits = (5 * (r64 / 64) * ((pixels + 255) / 256) >= 7 * cus && take(2, 2)) || take(2, 1);
  if (!fits && !take(1, 1)) return p;
  p.slab = p.rows * p.pitch;
  p.et = (2 * p.slab + NT - 1) / NT;
  if (p.st > 1 && p.et < 2) p.et = 2;   // (a kernel less)
  p.ctiles = (g->C + p.bm - 1) / p.bm;
  const long tiles = long(p.ctiles) * ((pixels + p.bn - 1) / p.bn);
  if (tiles >= (long(1) << 30)) return p;
  p.tiles = int(tiles);
  // Whole multiples of the CU count of tiles are one workgroup's each; the chunks of a remaining tile are dealt evenly to as
  // many workgroups as leave every CU at most one of them.  (Two per CU, or runs of chunks that cross tiles: more partial
  // tiles to write and sum, 64 images of 512 channels 7 x 7 93 against 92 / 101 us, of 128 channels 28 x 28 91 against 100 / 99.)
  p.dp_tiles = int(tiles / cus * cus);
  const int rest = p.tiles - p.dp_tiles;
  p.share = rest ? cus / rest : 1;
  if (p.share > p.nchunks) p.share = p.nchunks;
  if (p.share <= 1) p.share = 1, p.dp_tiles = p.tiles;
  p.wgs = p.dp_tiles + (p.tiles - p.dp_tiles) * p.share;
  p.weight_bytes = size_t(p.nchunks) * p.r * p.r * p.cblocks * kFrag;
  p.bytes = align256(p.weight_bytes) + size_t(p.wgs - p.dp_tiles) * p.bm * p.bn * sizeof(float);
  p.ok = true;
  return p;
}

namespace {

template <int GM, int WM, int WN, int ET, int R, int ST>
int launch(const ScArgs &a, const sgh_conv_split_plan &p, hipStream_t s) {
  auto kern = k_conv_split<GM, WM, WN, ET, R, ST>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) !=
        hipSuccess)
      return SGH_EUNSUPPORTED;
    attr_set = true;
  }
  SGH_LAUNCH_TIMED(kern, dim3(unsigned(p.wgs)), dim3(NT), size_t(p.slab) * 2 * kPos + 16, s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

// Weight fragments [chunk][tap][32-row block][part][lane][8]: one workgroup per (chunk, block).  Destination rows c are the
// output channels, k the reduction; the source is W[c][k][tap] (forward) or W[k][c][last - tap] (data gradient).
__global__ __launch_bounds__(256) void k_conv_split_weights(const float *__restrict__ W, uint16_t *__restrict__ wt, int C, int K,
                                                           int RS, int cblocks, int dgrad, int taps) {
  __shared__ float buf[kSplitWeightLds];
  sgh_conv_split_weights_block(W, wt, C, K, RS, cblocks, dgrad, int(blockIdx.x), taps, buf);
}

}  // namespace

int sgh_conv_split_weight_blocks(const sgh_conv_geom *g, int *cblocks, int *taps) {
  *cblocks = (g->C + 31) / 32;
  const int pairs = (g->K + KC - 1) / KC * *cblocks;
  *taps = pairs >= sgh_num_cus() ? kSplitTaps : kSplitTapsFew;
  return pairs * ((g->R * g->S + *taps - 1) / *taps);
}

int sgh_conv_split_weights(const sgh_conv_geom *g, const float *W, void *workspace, bool dgrad, hipStream_t s) {
  int cblocks, taps;
  const int blocks = sgh_conv_split_weight_blocks(g, &cblocks, &taps);
  hipLaunchKernelGGL(k_conv_split_weights, dim3(unsigned(blocks)), dim3(256), 0, s, W, static_cast<uint16_t *>(workspace), g->C,
                     g->K, g->R * g->S, cblocks, dgrad ? 1 : 0, taps);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

int sgh_conv_split_run(const sgh_conv_geom *g, const sgh_conv_split_plan &p, const float *in, const float *W, float *out, void *workspace,
                       hipStream_t s, const char *tag, bool dgrad, const float *bias, bool accumulate) {
  if (!p.ok) return SGH_EUNSUPPORTED;
  ScArgs a;
  a.in = in;
  a.W = W;
  a.w_c = (dgrad ? 1 : g->K) * p.r * p.r, a.w_k = (dgrad ? g->C : 1) * p.r * p.r;
  a.wt = static_cast<const uint16_t *>(workspace);
  a.bias = bias;
  a.out = out;
  a.partials = reinterpret_cast<float *>(static_cast<char *>(workspace) + align256(p.weight_bytes));
  a.accumulate = accumulate ? 1 : 0;
  a.dgrad = dgrad ? 1 : 0;
  a.N = g->N, a.C = g->C, a.K = g->K, a.P = g->P, a.Q = g->Q;
  a.IH = p.ih, a.IW = p.iw, a.plane = p.ih * p.iw * 4;
  a.cblocks = p.cblocks, a.pitch = p.pitch, a.slab = p.slab;
  a.total_pix = g->N * g->P * g->Q, a.nchunks = p.nchunks;
  a.ctiles = p.ctiles, a.dp_tiles = p.dp_tiles, a.share = p.share;
  a.xcd_runs = p.dp_tiles % 64 == 0 && !sgh_env().conv_xcd_off;
  a.in_bytes = unsigned(size_t(g->N) * g->K * p.ih * p.iw * 4);
  a.wt_bytes = unsigned(p.weight_bytes);
  int rc = SGH_EUNSUPPORTED;
  sgh_prof_kernel_begin(tag, 2.0 * g->N * g->K * g->P * g->Q * g->C * p.r * p.r);
#define SC_CASE(GM_, WM_, WN_, ET_, R_, ST_) \
  if (p.gm == GM_ && p.wm == WM_ && p.wn == WN_ && p.et == ET_ && p.r == R_ && p.st == ST_) rc = launch<GM_, WM_, WN_, ET_, R_, ST_>(a, p, s);
#define SC_CASES(GM_, WM_, WN_, R_) \
  SC_CASE(GM_, WM_, WN_, 1, R_, 1) SC_CASE(GM_, WM_, WN_, 2, R_, 1) SC_CASE(GM_, WM_, WN_, 3, R_, 1) SC_CASE(GM_, WM_, WN_, 4, R_, 1)
#define SC_CASES2(GM_, WM_, WN_) SC_CASE(GM_, WM_, WN_, 2, 3, 2) SC_CASE(GM_, WM_, WN_, 3, 3, 2)
  SC_CASES2(4, 1, 2)   // (256 pixels of stride 2 are more than 1024 places: no such tiles)
  SC_CASES2(2, 1, 1)
  SC_CASE(2, 1, 1, 4, 3, 2)
  SC_CASES(4, 1, 2, 3)
  SC_CASES(2, 1, 2, 3)
  SC_CASES(2, 1, 1, 3)
  SC_CASES(1, 1, 1, 3)
  SC_CASES(2, 1, 2, 5)
  SC_CASES(2, 1, 1, 5)
  SC_CASES(1, 1, 1, 5)
#undef SC_CASES2
#undef SC_CASES
#undef SC_CASE
  sgh_prof_kernel_end(s);
  if (rc != SGH_OK) return rc;
  if (p.share > 1) {
    hipLaunchKernelGGL(k_conv_split_fixup, dim3(unsigned(p.tiles - p.dp_tiles), unsigned(p.bm * p.bn / 1024)), dim3(256), 0, s, a,
                       p.bm, p.bn);
    if (hipGetLastError() != hipSuccess) return SGH_EINVAL;
  }
  return SGH_OK;
}
