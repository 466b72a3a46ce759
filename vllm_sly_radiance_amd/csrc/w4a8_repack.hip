// One-time repack of checkpoint MXFP4 weights into MFMA granules (layout in w4a8_internal.h).
//
// Replaces the reference's load-time permute_w + psw_pack_w_ + psw_fold_ws and the scale
// transpose (sly/mxfp4/radiance_mxfp4.py:181-226, :311-316, :1083-1171). On CDNA4 no nibble
// needs to move inside a byte and no exponent needs folding: a granule lane is 16 consecutive
// checkpoint bytes, so the weight repack is a permutation of 16-byte chunks and the scale repack
// a gather of single bytes into per-lane dwords. Padding (N to 16, K to 512) is zero nibbles with
// scale 127, which contributes exactly 0 to every output.
#include "w4a8_internal.h"

namespace w4a8 {
namespace {

constexpr int kThreads = 256;

// One thread per destination 16-byte chunk: coalesced 1 KiB granule writes.
__global__ __launch_bounds__(kThreads) void repack_nibbles(const uint8_t* __restrict__ w,
                                                          uint8_t* __restrict__ wq, int N, int K,
                                                          int KT, size_t total) {
  const size_t d = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (d >= total) return;
  const int lane = (int)(d & 63);
  const size_t g = d >> 6;
  const int kt = (int)(g % KT);
  const int nt = (int)(g / KT);
  const int n = nt * kNTile + (lane & 15);
  const int kb = kt * 4 + (lane >> 4);
  uint4 v = make_uint4(0, 0, 0, 0);
  if (n < N && kb < K / 32)
    v = *reinterpret_cast<const uint4*>(w + (size_t)n * (K / 2) + (size_t)kb * 16);
  reinterpret_cast<uint4*>(wq)[d] = v;
}

// One thread per destination scale dword: byte j = block (4 (4 kg + j) + lane / 16).
__global__ __launch_bounds__(kThreads) void repack_scales(const uint8_t* __restrict__ ws,
                                                         uint32_t* __restrict__ sq, int N, int K,
                                                         int KG, size_t total) {
  const size_t d = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (d >= total) return;
  const int lane = (int)(d & 63);
  const size_t g = d >> 6;
  const int kg = (int)(g % KG);
  const int nt = (int)(g / KG);
  const int n = nt * kNTile + (lane & 15);
  const int nb = K / 32;
  uint32_t v = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int kb = (kg * 4 + j) * 4 + (lane >> 4);
    const uint32_t e = (n < N && kb < nb) ? ws[(size_t)n * nb + kb] : 127u;
    v |= e << (8 * j);
  }
  sq[d] = v;
}

// Shapes with nothing to pad (N % 16 == 0, K % 512 == 0): one workgroup per n-tile, nibbles and
// scales in one launch, safe in place. An n-tile's 16 checkpoint rows and its granules are the same
// 8 K bytes (and its scale rows and scale dwords the same K / 2), so a workgroup that has read the
// whole stripe before one barrier may write it back where it came from: no second buffer and no copy
// back. The stripe's nibbles are a 16 x K / 32 matrix of 16-byte chunks and its granules the
// transpose: rows are read as whole KiB (wave w rows w and w + 8, every load in flight at once), put
// in LDS with a 16-byte row pad (a column's 16 chunks then lie in distinct banks) and stored as
// whole KiB granules. One row's 16 scale bytes of one k-group are a 4 x 4 byte transpose of a
// column of 4 dwords. Bound by memory, one read and one write of the layer: N = 17408 K = 5120 15.3 us
// on MI355X (95 MB, 6.2 TB/s) against 15.1 + 8.2 us for the general kernels and two copies back
// (12 us more); with 64-byte gathers of 16 rows straight to registers instead of the LDS rows 24.7.
// One layer's load (four projections, the checkpoint copies included) 209 -> 148 us. V: 64-chunk loads per row, K <= 2048 V.
constexpr int kStripeThreads = 512;
constexpr int kStripeMaxK = 19968;               // 16 padded rows within 160 KiB of LDS

int stripe_lds(int K) { return kNTile * (K / 2 + 16); }

template <int V>
__global__ __launch_bounds__(kStripeThreads) void repack_stripe(const uint8_t* w, const uint8_t* ws,
                                                                uint8_t* wq, uint32_t* sq, int K) {
  extern __shared__ __attribute__((aligned(16))) uint8_t rows[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int RB = K >> 1, KG = K / kKAlign, pitch = RB + 16;
  const size_t stripe = (size_t)blockIdx.x * kNTile * RB;
  const auto src = __builtin_amdgcn_make_buffer_rsrc((void*)(w + stripe), 0, kNTile * RB,
                                                     kBufferWord3);
  const uint8_t* const sr = ws + (size_t)blockIdx.x * kNTile * (K / 32);
  uint32_t* const sd = sq + (size_t)blockIdx.x * KG * 64;
  const int r = tid & 15, kg0 = tid >> 4;        // scale items (kg, r), 32 k-groups per pass
  uint4 sv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int kg = kg0 + 32 * i;
    if (kg < KG) sv[i] = *reinterpret_cast<const uint4*>(sr + (size_t)r * (K / 32) + kg * 16);
  }
  v4i v[2][V];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int at = (lane + 64 * i) * 16;       // past the row: no access, zeros
      v[h][i] = __builtin_amdgcn_raw_buffer_load_b128(
          src, at < RB ? (wave + 8 * h) * RB + at : 0x7FFFFFF0, 0, 0);
    }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int at = (lane + 64 * i) * 16;
      if (at < RB) *reinterpret_cast<v4i*>(rows + (wave + 8 * h) * pitch + at) = v[h][i];
    }
  // every load of the stripe, scales too, has returned in every wave before any store to it
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  v4i* const wd = reinterpret_cast<v4i*>(wq + stripe);
  for (int d = tid; d < RB; d += kStripeThreads)           // RB chunks of 16 bytes
    wd[d] = *reinterpret_cast<const v4i*>(rows + (d & 15) * pitch + (d >> 4) * 16);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int kg = kg0 + 32 * i;
    if (kg >= KG) continue;
    // dword q: byte j = the row's block 4 j + q of the k-group, that is byte q of its dword j
    const uint32_t a[4] = {sv[i].x, sv[i].y, sv[i].z, sv[i].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t o = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) o |= ((a[j] >> (8 * q)) & 0xFFu) << (8 * j);
      sd[kg * 64 + q * 16 + r] = o;
    }
  }
}

}  // namespace

bool repack_in_place(const uint8_t* ws, int N, int K) {
  return N % kNTile == 0 && K % kKAlign == 0 && K <= kStripeMaxK && ((uintptr_t)ws % 16) == 0;
}

hipError_t launch_repack(const uint8_t* w, const uint8_t* ws, uint8_t* wq, uint32_t* sq, int N,
                         int K, hipStream_t stream) {
  const int NT = padded_n(N) / kNTile, KT = padded_k(K) / kKTile, KG = KT / kKGroup;
  const size_t chunks = (size_t)NT * KT * 64, dwords = (size_t)NT * KG * 64;
  if (chunks == 0) return hipSuccess;
  if (repack_in_place(ws, N, K)) {
    const int lds = stripe_lds(K);
#define W4A8_STRIPE(V)                                                                           \
  if (K <= 2048 * V) {                                                                           \
    if (lds > 64 * 1024) {                                                                       \
      const hipError_t e = hipFuncSetAttribute((const void*)repack_stripe<V>,                    \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
      if (e != hipSuccess) return e;                                                             \
    }                                                                                            \
    hipLaunchKernelGGL((repack_stripe<V>), dim3(NT), dim3(kStripeThreads), lds, stream, w, ws,   \
                       wq, sq, K);                                                               \
    return hipGetLastError();                                                                    \
  }
    W4A8_STRIPE(1) W4A8_STRIPE(2) W4A8_STRIPE(3) W4A8_STRIPE(5) W4A8_STRIPE(10)
#undef W4A8_STRIPE
  }
  hipLaunchKernelGGL(repack_nibbles, dim3((unsigned)((chunks + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, stream, w, wq, N, K, KT, chunks);
  hipLaunchKernelGGL(repack_scales, dim3((unsigned)((dwords + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, stream, ws, sq, N, K, KG, dwords);
  return hipGetLastError();
}

}  // namespace w4a8
