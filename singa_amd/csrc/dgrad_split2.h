// fp32 data gradient of 3x3 convolutions of stride 2 on split operands (dgrad_split2.hip)
#ifndef SINGA_AMD_CSRC_DGRAD_SPLIT2_H_
#define SINGA_AMD_CSRC_DGRAD_SPLIT2_H_

#include "common.h"
#include "split_parts.h"

bool sgh_dgrad_split2_supported(const sgh_conv_geom *g);
// weight fragments (the ones of conv_split.h, as for a data gradient), then the partial tiles
size_t sgh_dgrad_split2_workspace_bytes(const sgh_conv_geom *g);
int sgh_dgrad_split2_run(const sgh_conv_geom *g, const float *dy, const float *W, float *dx, void *workspace, hipStream_t s,
                         bool accumulate);

#endif  // SINGA_AMD_CSRC_DGRAD_SPLIT2_H_
