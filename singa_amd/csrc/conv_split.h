// fp32 convolutions on split operands (conv_split.hip): "same" padding, 3x3 and 5x5 of stride 1 and forward passes of 3x3 and stride 2.
// `g` is the geometry of the data gradient: K channels of `in` are gathered onto C channels of `out`; a forward pass hands in the
// channel-swapped one.
#ifndef SINGA_AMD_CSRC_CONV_SPLIT_H_
#define SINGA_AMD_CSRC_CONV_SPLIT_H_

#include "common.h"
#include "split_parts.h"

// How the layer runs; made once per call (stride 2: a microsecond of host time)
struct sgh_conv_split_plan {
  bool ok;   // false: a layer for other kernels
  int r, st, gm, wm, wn, et, bm, bn, ih, iw, pitch, rows, slab, nchunks, cblocks;
  int ctiles, tiles, dp_tiles, share, wgs;
  size_t weight_bytes, bytes;   // of the workspace: the weight fragments, and with the partial tiles behind them
};
sgh_conv_split_plan sgh_conv_split_plan_of(const sgh_conv_geom *g);
// the weight fragments of `g` into the front of `workspace`, from W[C][K][R][S] or (dgrad) W[K][C][R][S]
int sgh_conv_split_weights(const sgh_conv_geom *g, const float *W, void *workspace, bool dgrad, hipStream_t s);
// the same as a batch item: workgroups of sgh_conv_split_weights_block
int sgh_conv_split_weight_blocks(const sgh_conv_geom *g, int *cblocks, int *taps);
// `W`: the same weights again, for what the fragments cannot hold
int sgh_conv_split_run(const sgh_conv_geom *g, const sgh_conv_split_plan &p, const float *in, const float *W, float *out, void *workspace,
                       hipStream_t s, const char *tag, bool dgrad, const float *bias, bool accumulate);

constexpr int kSplitWeightLds = 512 * 9;   // floats of LDS that a workgroup below needs

// Taps that a workgroup below handles: all of a small filter once that many workgroups fill the chip, else a third of them (64 to
// 64 channels, eight (chunk, block) pairs: 8.1 -> 4.9 us, the time of three rounds of loads)
constexpr int kSplitTaps = 9, kSplitTapsFew = 3;

// One (chunk of 16 channels k, block of 32 channels c) of the weight fragments [chunk][tap][block][part][lane][8], by 256
// threads: the source runs are contiguous, the fragments too, LDS turns one into the other.
// w0 + w1 + w2 is kSplitScale w, or not finite where that does not fit; odd taps are negated.
__device__ __forceinline__ void sgh_conv_split_weights_block(const float *__restrict__ W, uint16_t *__restrict__ wt, int C, int K,
                                                             int RS, int cblocks, int dgrad, int blk, int taps, float *buf) {
  const int groups = (RS + taps - 1) / taps, group = blk % groups;
  blk /= groups;
  const int ch = blk / cblocks, cb = blk - ch * cblocks, k0 = ch * 16, c0 = cb * 32, t = threadIdx.x;
  {
    const int t0 = group * taps, nt = RS - t0 < taps ? RS - t0 : taps, total = 512 * nt, inner = dgrad ? 32 : 16;
    constexpr int U = 6;
    for (int i0 = t; i0 < total; i0 += 256 * U) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * 256, row = i / nt, tap = i - row * nt, a = row / inner, b = row - a * inner;
        const int c = c0 + (dgrad ? b : a), k = k0 + (dgrad ? a : b);
        const bool ok = i < total && c < C && k < K;
        v[u] = ok ? W[(dgrad ? long(k) * C + c : long(c) * K + k) * RS + t0 + tap] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * 256, row = i / nt, tap = i - row * nt, a = row / inner, b = row - a * inner;
        if (i < total) buf[((dgrad ? b : a) * 16 + (dgrad ? a : b)) * 9 + tap] = v[u];   // [c][k][tap]
      }
    }
    __syncthreads();
    for (int i = t; i < 64 * nt; i += 256) {
      const int tap = i >> 6, lane = i & 63;
      const float *src = buf + ((lane & 31) * 16 + (lane >> 5) * 8) * 9 + tap;
      const int q = ch * RS + (dgrad ? RS - 1 - (t0 + tap) : t0 + tap);
      uint16_t part[3][8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const Parts w = split2(q % RS & 1 ? -src[j * 9] : src[j * 9], 0.f);
        part[0][j] = uint16_t(w.p[0]), part[1][j] = uint16_t(w.p[1]), part[2][j] = uint16_t(w.p[2]);
      }
      uint16_t *dst = wt + (size_t(q) * cblocks + cb) * 1536 + lane * 8;
#pragma unroll
      for (int p = 0; p < 3; ++p) __builtin_memcpy(dst + p * 512, part[p], 16);
    }
  }
}

#endif  // SINGA_AMD_CSRC_CONV_SPLIT_H_
