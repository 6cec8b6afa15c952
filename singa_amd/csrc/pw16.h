// 1x1 / stride 1 / unpadded convolutions on 16-bit tensors (pw16.hip); called by the plans of conv16.hip.
#ifndef SINGA_AMD_CSRC_PW16_H_
#define SINGA_AMD_CSRC_PW16_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

struct sgh_pw16_args {
  const uint16_t *A;     // [M][lda]: filters, reduction index contiguous; zero (or beyond the buffer) outside M x K
  const uint16_t *src;   // [N][K][HW]
  uint16_t *out;         // [N][M][HW]
  const uint16_t *bias;  // per output channel, or null
  const uint16_t *add, *gate;   // out = gate > 0 ? stored result + add : 0, both laid out as out; or null
  int M, K, HW, lda;     // K and lda: multiples of 8, HW >= 8
  int QO, octets;        // octets of a plane (the last one overlaps its neighbour), of the batch
  int mtiles, ptiles;
  unsigned a_bytes, src_bytes;
};

int sgh_pw16_tile(int M, long ptiles);   // filters per workgroup: 64, 128 or 256
int sgh_pw16_launch(sgh_pw16_args a, int bm, bool bf16, hipStream_t s);

#endif  // SINGA_AMD_CSRC_PW16_H_
