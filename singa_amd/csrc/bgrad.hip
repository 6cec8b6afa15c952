// Bias gradient of a convolution: db[k] = sum over images and pixels of dy[n][k][p][q].
//
// Bound by reading dy once.  The entry points take no workspace and the sum of a channel has to come out the same on
// every run, so one workgroup owns a channel; with 64 channels three quarters of the CUs stay idle and the kernel is
// only as fast as one CU can pull bytes: 1024 threads with eight 16-byte loads in flight each (128 KB per CU).
// 64 x 64 x 56 x 56 fp32 (51 MB): 265 us before (256 threads, one dword in flight, a division per element), 12 us.
#include "common.h"
#include "storage.h"

namespace {

constexpr int BT = 1024, BU = 8;

typedef __amdgpu_buffer_rsrc_t rsrc_t;

// A piece of 16 bytes, or one element of 4 or 2 bytes (planes shorter than a vector), at element alignment
template <int BYTES>
struct Piece;
template <>
struct Piece<16> {
  typedef unsigned int type __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ type ld(rsrc_t r, int off) { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0); }
};
template <>
struct Piece<4> {
  typedef unsigned int type __attribute__((ext_vector_type(1)));
  static __device__ __forceinline__ type ld(rsrc_t r, int off) { return type{__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0)}; }
};
template <>
struct Piece<2> {
  typedef unsigned short type __attribute__((ext_vector_type(1)));
  static __device__ __forceinline__ type ld(rsrc_t r, int off) { return type{__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0)}; }
};

// V elements of the storage class per piece: S::VEC, or 1 for planes shorter than that.  A plane that is not a whole
// number of pieces ends with a piece that starts at PQ - V: its first V - PQ mod V elements belong to the piece before.
template <class S, int V, bool RAGGED>
__global__ __launch_bounds__(BT) void k_conv_bgrad(const typename S::elem *__restrict__ dy, typename S::elem *__restrict__ db,
                                                   int N, int K, int PQ, unsigned bytes) {
  typedef typename S::elem elem;
  typedef Piece<V * int(sizeof(elem))> P;
  __shared__ float red[16];
  const int k = blockIdx.x, t = threadIdx.x;
  const rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(const_cast<elem *>(dy), 0, bytes, 0x00020000);
  const int VP = (PQ + V - 1) / V;               // pieces per plane
  const int dn = BT / VP, dv = BT - dn * VP;     // a step of BT pieces: images, and pieces within a plane
  const int back = RAGGED ? VP * V - PQ : 0;
  int n = t / VP, v = t - n * VP;
  float acc[BU];
#pragma unroll
  for (int u = 0; u < BU; ++u) acc[u] = 0.f;
  while (n < N) {
    typename P::type r[BU];
    bool last[BU];
#pragma unroll
    for (int u = 0; u < BU; ++u) {
      last[u] = RAGGED && v == VP - 1;
      const int first = v * V - (last[u] ? back : 0);
      // (past the end: an offset the buffer refuses, which yields zeros)
      r[u] = P::ld(src, n < N ? ((n * K + k) * PQ + first) * int(sizeof(elem)) : int(0x80000000u));
      n += dn, v += dv;
      if (v >= VP) v -= VP, ++n;
    }
#pragma unroll
    for (int u = 0; u < BU; ++u) {
      elem e[V];
      __builtin_memcpy(e, &r[u], sizeof(e));
      float f[V];
#pragma unroll
      for (int j = 0; j < V; ++j) f[j] = RAGGED && last[u] && j < back ? 0.f : S::ld(e + j);
#pragma unroll
      for (int w = V / 2; w > 0; w /= 2)
#pragma unroll
        for (int j = 0; j < w; ++j) f[j] += f[j + w];
      acc[u] += f[0];
    }
  }
#pragma unroll
  for (int w = BU / 2; w > 0; w /= 2)
#pragma unroll
    for (int u = 0; u < w; ++u) acc[u] += acc[u + w];
  const float s = sgh_block_sum(acc[0], red);
  if (t == 0) S::st(db + k, s);
}

template <class S>
int run(const sgh_conv_geom *g, const void *dy, void *db, hipStream_t s) {
  typedef typename S::elem elem;
  const int PQ = g->P * g->Q;
  const unsigned bytes = unsigned(size_t(g->N) * g->K * PQ * sizeof(elem));
  const elem *src = static_cast<const elem *>(dy);
  elem *dst = static_cast<elem *>(db);
  if (PQ < S::VEC) hipLaunchKernelGGL((k_conv_bgrad<S, 1, false>), dim3(g->K), dim3(BT), 0, s, src, dst, g->N, g->K, PQ, bytes);
  else if (PQ % S::VEC) hipLaunchKernelGGL((k_conv_bgrad<S, S::VEC, true>), dim3(g->K), dim3(BT), 0, s, src, dst, g->N, g->K, PQ, bytes);
  else hipLaunchKernelGGL((k_conv_bgrad<S, S::VEC, false>), dim3(g->K), dim3(BT), 0, s, src, dst, g->N, g->K, PQ, bytes);
  SGH_LAUNCH_CHECK();
  return SGH_OK;
}

}  // namespace

int sgh_conv_bgrad_run(const sgh_conv_geom *g, const void *dy, void *db, int dtype, hipStream_t s) {
  return dtype == 0 ? run<StF32>(g, dy, db, s) : dtype == 1 ? run<StF16>(g, dy, db, s) : run<StBF16>(g, dy, db, s);
}
