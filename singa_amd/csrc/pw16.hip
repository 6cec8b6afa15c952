// 1x1 / stride 1 / unpadded convolutions on 16-bit NCHW tensors, forward and data gradient:
//   out[n][m][pix] = sum_k A[m][k] * src[n][k][pix]      (v_mfma_f32_32x32x16_{f16,bf16}, fp32 accumulation)
// with A the filters ([m][k], k contiguous: the weight tensor itself in the forward pass, its transposed copy in the
// data gradient).  The reduction index is the strided one of `src` while the matrix instructions want eight
// consecutive reduction indices per lane.  The tile is kept as it lies in memory, [k][pixel], and the transposition
// happens where the fragments are read: ds_read_b64_tr_b16 hands a lane four k of its pixel.  So a tile of `src` is
// staged by 16-byte loads that write LDS themselves, with no register, no permutation and no LDS store in between.
// Pixels are independent columns: a plane is cut into octets, the last of which ends with the plane and overlaps its
// neighbour (both compute and store the same bits), so any plane of eight pixels or more works without masks.
//   Pipeline: a ring of ST chunks of KC reduction indices, ST - 1 of them on their way while one is multiplied, one
// barrier per chunk, two workgroups per CU.  Every request is issued unconditionally (one beyond the reduction goes
// out of range and writes zeros into a free slot), so the wait counts loads instead of draining them.
//   LDS layout: 16-byte slots.  A slot of `src` row k sits at octet ^ ((k & 3) << 2): the four k rows of a transposing
// read then cover all banks.  A filter row's octets are rotated the same way by the row index.
//   Bound by bytes on large planes, by the reads from L2 on small ones.  Forward, binary16, against dword loads and
// permutations in registers (and a copy of the filters): 128 x 64 x 56 x 56 -> 256 76.5 -> 49.2 us (5.2 TB/s),
// 128 x 1024 x 14 x 14 -> 256 31.2 -> 23.3, 21 x 2048 x 6 x 6 -> 512 31.7 -> 14.2.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "pw16.h"
#include "storage.h"

namespace {

constexpr int NT = 512, BN = 128;   // threads; pixels of a tile (16 octets)
constexpr int kOOB = int(0x80000000u);

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

template <bool BF16>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Transposing reads: within each 16 lanes, lane i addresses four pixels of k row i / 4 and receives pixel i of all four
// rows.  A pair of them (k and k + 4) is an operand of one matrix instruction; p0 / p1 are the bases of two columns of
// steps, `out` receives the steps at +0 and +16 rows of each.  One block with its own wait: the builtin makes the
// compiler drain every request to LDS that is under way before it (here vmcnt(0) per chunk, i.e. no pipeline).
template <int COLS>
__device__ __forceinline__ void read_tr(const uint16_t *p0, const uint16_t *p1, u32x4 (&out)[COLS][2]) {
  typedef __attribute__((address_space(3))) const uint16_t lds_u16;
  const unsigned a0 = unsigned(size_t((lds_u16 *)p0));
  u32x2 r[8];
  static_assert(BN == 128, "immediates: 4 rows = 1024 bytes, 16 rows = 4096");
  if constexpr (COLS == 2) {
    const unsigned a1 = unsigned(size_t((lds_u16 *)p1));
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:1024\n\t"
        "ds_read_b64_tr_b16 %4, %9\n\tds_read_b64_tr_b16 %5, %9 offset:1024\n\t"
        "ds_read_b64_tr_b16 %2, %8 offset:4096\n\tds_read_b64_tr_b16 %3, %8 offset:5120\n\t"
        "ds_read_b64_tr_b16 %6, %9 offset:4096\n\tds_read_b64_tr_b16 %7, %9 offset:5120\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
        : "v"(a0), "v"(a1)
        : "memory");
  } else {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %4 offset:1024\n\t"
        "ds_read_b64_tr_b16 %2, %4 offset:4096\n\tds_read_b64_tr_b16 %3, %4 offset:5120\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(a0)
        : "memory");
  }
#pragma unroll
  for (int j = 0; j < COLS; ++j)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      out[j][k] = u32x4{r[4 * j + 2 * k][0], r[4 * j + 2 * k][1], r[4 * j + 2 * k + 1][0], r[4 * j + 2 * k + 1][1]};
}

template <int BM, int KC, int ST>
constexpr int pw_stage_halves() { return (BM + BN) * KC; }

// BM filters x 128 pixels per workgroup, eight wavefronts of (32 * TM) x (32 * TN).
// DMA: `src` and its rows are dword aligned (even planes): loads write LDS; otherwise octets at any element
// alignment go through two register sets, two chunks ahead.
template <int BM, int KC, int ST, bool BF16, bool DMA>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_pw16(sgh_pw16_args a) {
  constexpr int WM = BM / 64 == 1 ? 2 : (BM == 128 ? 2 : 4), WN = 8 / WM;
  constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN);
  constexpr int NA = BM * KC / (8 * NT), NB = BN * KC / (8 * NT), OPR = KC / 8;   // loads per thread and chunk
  constexpr int STAGE = pw_stage_halves<BM, KC, ST>(), BOFF = BM * KC;
  static_assert(NA >= 1 && NB >= 1 && ST >= 3, "");
  extern __shared__ __align__(16) uint16_t lds[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN, l32 = lane & 31, lh = lane >> 5;
  // workgroup w runs on XCD w % 8: the filter tiles of one pixel tile read the same pixels through one L2
  const int slot = int(blockIdx.x) >> 3, pt = (slot / a.mtiles) * 8 + (int(blockIdx.x) & 7);
  if (pt >= a.ptiles) return;
  const int m0 = (slot % a.mtiles) * BM;
  const rsrc_t ra = make_rsrc(a.A, a.a_bytes), rs = make_rsrc(a.src, a.src_bytes);

  // filters: 16-byte slot j * NT + t of the tile -> row, octet
  const int arow = t / OPR, aoct = (t % OPR) ^ (OPR == 4 ? (arow >> 2) & 3 : (arow >> 1) & 7);
  const int avoff = ((m0 + arow) * a.lda + aoct * 8) * 2, astep = NT / OPR * a.lda * 2;
  // pixels: row k = 32 j + t / 16, octet of the tile
  const int bk = t >> 4, boct = (t & 15) ^ ((bk & 3) << 2);
  int bvoff = kOOB;
  {
    const int go = pt * 16 + boct;
    if (go < a.octets) {
      const int n = go / a.QO, p = go - n * a.QO;
      bvoff = ((n * a.K + bk) * a.HW + min(8 * p, a.HW - 8)) * 2;
    }
  }
  const int bstep = 32 * a.HW * 2;
  const int nch = (a.K + KC - 1) / KC;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // fragment addresses: filter row and its octet rotation; pixel column of a transposing read
  const int frow = wm * TM * 32 + l32, fswz = OPR == 4 ? (frow >> 2) & 3 : (frow >> 1) & 7;
  const int trk = 8 * lh + ((lane >> 2) & 3), trs = ((lane >> 2) & 3) << 2;
  const int trlow = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
  auto multiply = [&](const uint16_t *st) {
#pragma unroll
    for (int k0 = 0; k0 < KC / 16; k0 += 2) {   // two matrix steps at a time
      u32x4 fa[TM][2], fb[TN][2];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k)
          fa[i][k] = *reinterpret_cast<const u32x4 *>(st + (frow + 32 * i) * KC + ((2 * (k0 + k) + lh) ^ fswz) * 8);
      const uint16_t *b = st + BOFF + (16 * k0 + trk) * BN + (lane & 1) * 4;
      read_tr<TN>(b + (((4 * (wn * TN)) ^ trs) + trlow) * 8, b + (((4 * (wn * TN + TN - 1)) ^ trs) + trlow) * 8, fb);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = mfma<BF16>(fb[j][k], fa[i][k], acc[i][j]);   // rows: pixels, columns: filters
    }
  };

  if constexpr (DMA) {
    typedef __attribute__((address_space(3))) void lds_void;
    auto request = [&](int c, int s) {
      uint16_t *st = lds + s * STAGE + wave * 512;
      const int ao = c < nch ? avoff : kOOB;
#pragma unroll
      for (int j = 0; j < NA; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void *)(st + j * NT * 8), 16, c < nch ? ao + j * astep : kOOB, c * KC * 2, 0, 0);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(st + BOFF + j * NT * 8), 16,
                                                 c * KC + 32 * j + bk < a.K && bvoff != kOOB ? bvoff + j * bstep : kOOB, c * KC * a.HW * 2, 0, 0);
    };
#pragma unroll
    for (int c = 0; c < ST - 1; ++c) request(c, c);
    int s = 0;
    for (int c = 0; c < nch; ++c) {
      // chunk c has arrived (the ST - 2 newer ones may be under way) and everybody is done with the slot before it
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((ST - 2) * (NA + NB)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      request(c + ST - 1, s == 0 ? ST - 1 : s - 1);
      multiply(lds + s * STAGE);
      s = s + 1 == ST ? 0 : s + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last requests write zeros)
  } else {
    u32x4 va[2][NA], vb[2][NB];
    auto request = [&](auto SET, int c) {
      constexpr int S = decltype(SET)::value;
#pragma unroll
      for (int j = 0; j < NA; ++j)
        va[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, c < nch ? avoff + j * astep : kOOB, c * KC * 2, 0));
#pragma unroll
      for (int j = 0; j < NB; ++j)
        vb[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
            rs, c * KC + 32 * j + bk < a.K && bvoff != kOOB ? bvoff + j * bstep : kOOB, c * KC * a.HW * 2, 0));
    };
    auto stage = [&](auto SET, uint16_t *st) {
      constexpr int S = decltype(SET)::value;
#pragma unroll
      for (int j = 0; j < NA; ++j) *reinterpret_cast<u32x4 *>(st + (j * NT + t) * 8) = va[S][j];
#pragma unroll
      for (int j = 0; j < NB; ++j) *reinterpret_cast<u32x4 *>(st + BOFF + (j * NT + t) * 8) = vb[S][j];
    };
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    uint16_t *const st0 = lds, *const st1 = lds + STAGE;
    request(Set0{}, 0);
    request(Set1{}, 1);
    stage(Set0{}, st0);
    for (int c = 0;; c += 2) {
      __syncthreads();
      request(Set0{}, c + 2);
      multiply(st0);
      if (c + 1 >= nch) break;
      stage(Set1{}, st1);
      __syncthreads();
      request(Set1{}, c + 3);
      multiply(st1);
      if (c + 2 >= nch) break;
      stage(Set0{}, st0);
    }
  }

  // the tile leaves through LDS as [filter][pixel] rows; a lane holds four neighbouring pixels of one filter
  constexpr int OP = BN + 8;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = frow + 32 * i;
    float bias = 0.f;
    if (a.bias && m0 + row < a.M) bias = BF16 ? sgh_bf16_to_f32(a.bias[m0 + row]) : sgh_f16_to_f32(a.bias[m0 + row]);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; v += 4) {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = a.bias ? acc[i][j][v + e] + bias : acc[i][j][v + e];
        const u32x2 o = BF16 ? u32x2{sgh_pack2_bf16(x[0], x[1]), sgh_pack2_bf16(x[2], x[3])}
                             : u32x2{sgh_pack2_f16(x[0], x[1]), sgh_pack2_f16(x[2], x[3])};
        *reinterpret_cast<u32x2 *>(lds + row * OP + (wn * TN + j) * 32 + 2 * v + 4 * lh) = o;
      }
  }
  const int g = t & 15, go = pt * 16 + g;
  const int n = go / a.QO, p = go - n * a.QO;
  const size_t first = (size_t(n) * a.M + m0) * a.HW + min(8 * p, a.HW - 8);
  // A residual block's input gradient: the sum with its other branch and the ReLU in front of the block.  Two reads here instead of
  // a pass of its own that reads three tensors and writes one (ResNet-50, 128 images: 0.85 of 13.2 ms of kernel time).  Both are
  // requested before the tile is complete.
  if (a.add) {
    u32x4 va[BM / 32], vg[BM / 32];
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      const int row = (t >> 4) + 32 * i;
      if (go < a.octets && m0 + row < a.M) {
        __builtin_memcpy(&va[i], a.add + first + size_t(row) * a.HW, 16);
        __builtin_memcpy(&vg[i], a.gate + first + size_t(row) * a.HW, 16);
      }
    }
    __syncthreads();
    if (go >= a.octets) return;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      const int row = (t >> 4) + 32 * i;
      if (m0 + row >= a.M) continue;
      const u32x4 v = *reinterpret_cast<const u32x4 *>(lds + row * OP + 8 * g);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float r[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          auto value = [&](const u32x4 &w) {
            const uint16_t b = uint16_t(w[e] >> (16 * k));
            return BF16 ? sgh_bf16_to_f32(b) : sgh_f16_to_f32(b);
          };
          r[k] = value(vg[i]) > 0.f ? value(v) + value(va[i]) : 0.f;
        }
        o[e] = BF16 ? sgh_pack2_bf16(r[0], r[1]) : sgh_pack2_f16(r[0], r[1]);
      }
      __builtin_memcpy(a.out + first + size_t(row) * a.HW, &o, 16);
    }
    return;
  }
  __syncthreads();
  if (go >= a.octets) return;
#pragma unroll
  for (int i = 0; i < BM / 32; ++i) {
    const int row = (t >> 4) + 32 * i;
    if (m0 + row < a.M) __builtin_memcpy(a.out + first + size_t(row) * a.HW, lds + row * OP + 8 * g, 16);
  }
}

template <int BM, int KC, int ST, bool BF16, bool DMA>
int launch(const sgh_pw16_args &a, hipStream_t s) {
  auto kern = k_pw16<BM, KC, ST, BF16, DMA>;
  constexpr int ring = (DMA ? ST : 2) * pw_stage_halves<BM, KC, ST>(), tile = BM * (BN + 8);
  constexpr size_t bytes = size_t(ring > tile ? ring : tile) * 2;
  static bool allowed = false;
  if (!allowed) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)) != hipSuccess)
      return SGH_EUNSUPPORTED;
    allowed = true;
  }
  SGH_LAUNCH_TIMED(kern, dim3(unsigned((a.ptiles + 7) / 8) * 8u * unsigned(a.mtiles)), dim3(NT), bytes, s, a);
  return hipGetLastError() == hipSuccess ? SGH_OK : SGH_EINVAL;
}

template <int BM, int KC, int ST>
int launch_typed(const sgh_pw16_args &a, bool bf16, bool dma, hipStream_t s) {
  if (dma) return bf16 ? launch<BM, KC, ST, true, true>(a, s) : launch<BM, KC, ST, false, true>(a, s);
  return bf16 ? launch<BM, KC, ST, true, false>(a, s) : launch<BM, KC, ST, false, false>(a, s);
}

}  // namespace

// The largest tile that still gives three quarters of the CUs a workgroup: its operands are read least often, but with
// fewer workgroups the CUs that are left out cost more.  us for 64 / 128 / 256 filters, binary16: forward
// 128 x 1024 x 14 x 14 -> 256 28.4 / 26.5 / 23.3 (800 / 400 / 200 workgroups), 21 x 512 x 24 x 24 -> 128 6.2 / 8.4
// (190 / 95), 21 x 1024 x 12 x 12 -> 256 8.7 / 12.7 / 17.7 (96 / 48 / 24).
int sgh_pw16_tile(int M, long ptiles) {
  const long enough = sgh_num_cus() * 3 / 4;
  if (M > 128 && ptiles * ((M + 255) / 256) >= enough) return 256;
  return M > 64 && ptiles * ((M + 127) / 128) >= enough ? 128 : 64;
}

int sgh_pw16_launch(sgh_pw16_args a, int bm, bool bf16, hipStream_t s) {
  const bool dma = a.HW % 2 == 0 && ((reinterpret_cast<uintptr_t>(a.src) | reinterpret_cast<uintptr_t>(a.A)) & 3u) == 0;
  if (bm == 64) return launch_typed<64, 64, 3>(a, bf16, dma, s);
  if (bm == 256 && dma) return bf16 ? launch<256, 32, 3, true, true>(a, s) : launch<256, 32, 3, false, true>(a, s);
  a.mtiles = (a.M + 127) / 128;   // (the register path has no room for the accumulators of 256 filters)
  return launch_typed<128, 32, 4>(a, bf16, dma, s);
}
