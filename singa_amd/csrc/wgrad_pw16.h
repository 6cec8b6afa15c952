// Weight gradients of 1x1 / stride 1 / unpadded convolutions on 16-bit tensors (wgrad_pw16.hip); called by conv16.hip.
#ifndef SINGA_AMD_CSRC_WGRAD_PW16_H_
#define SINGA_AMD_CSRC_WGRAD_PW16_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "singa_hip.h"

struct sgh_wgrad_pw16_plan {
  bool ok;
  int bm, bn;                            // filters x channels of a tile
  int tiles, parts, chunks, per_part;    // parts of the reduction; chunks of 64 pixels, of one part
};

sgh_wgrad_pw16_plan sgh_wgrad_pw16_plan_of(const sgh_conv_geom *g);
// One partial image [K][C] per part into `partial`, or dW itself when there is one part
int sgh_wgrad_pw16_run(const sgh_conv_geom *g, const sgh_wgrad_pw16_plan &p, const uint16_t *dy, const uint16_t *x, float *partial,
                       uint16_t *dW, bool bf16, hipStream_t s);

#endif  // SINGA_AMD_CSRC_WGRAD_PW16_H_
