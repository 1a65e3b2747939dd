// Layout conversions at the model boundary for gfx950: NCHW float32 images ->
// NHWC element-type rows (zero-padded channels), and back.
//
// Both are copies, so HBM bounds them; what has to be arranged is that both
// sides are read and written in whole lines although one has the pixels and
// the other the channels next to each other.  A workgroup takes CT channels x
// PT pixels of one image (4096 values) through LDS as [channel][pixel] rows of
// PT + 1 floats: the float32 side moves 4 pixels of one channel per lane, the
// NHWC side one 16-byte chunk of a pixel per lane with the chunks of a pixel
// on neighbouring lanes (64 channels of bfloat16 = one 128-byte line); the odd
// row length keeps both accesses of LDS off each other's banks.  Measured:
// 512 channels x 20x20 x 32 images to bfloat16 (39 MB) 195 us with one thread
// per pixel (4 workgroup rounds of 512 dependent strided stores) -> 6.9 us;
// back 30 us (one thread per value, 2-byte loads a pixel apart) -> 6.9 us (5.7 TB/s, in the cache).
#include "common.h"

namespace {

template <typename T, int CT>
__device__ __forceinline__ bool layout_tile(const vrs_pack_args& a, int& b, int& c0, int64_t& p0) {
  constexpr int PT = 4096 / CT;
  const int logical = xcd_remap(blockIdx.x, gridDim.x);
  const int tc = logical % a.tiles_c, r = logical / a.tiles_c;
  c0 = tc * CT;
  b = r / a.tiles_p;
  p0 = (int64_t)(r - b * a.tiles_p) * PT;
  return b < a.N;
}

template <typename T, int CT>
__device__ __forceinline__ void pack_body(const vrs_pack_args& a) {
  constexpr int PT = 4096 / CT, ROW = PT + 1, PQ = PT / 4;
  constexpr int EPC = 16 / (int)sizeof(T), CPP = CT / EPC;   // elements per chunk, chunks per pixel
  __shared__ float tile[CT * ROW];
  int b, c0;
  int64_t p0;
  if (!layout_tile<T, CT>(a, b, c0, p0)) return;
  const float* x = reinterpret_cast<const float*>(a.x) + ((int64_t)b * a.C + c0) * a.HW + p0;
  T* y = reinterpret_cast<T*>(a.y) + ((int64_t)b * a.HW + p0) * a.c_pad + c0;
  const int np = (int)min((int64_t)PT, a.HW - p0), nc = min(CT, a.C - c0);   // valid pixels and (may be <= 0) channels
  const int tid = threadIdx.x;
  f32x4_t v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = tid + i * 256, c = t / PQ, q = t % PQ;
    v[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (c < nc && 4 * q < np) {
      const float* s = x + (int64_t)c * a.HW + 4 * q;
      if (a.vec_p) {   // HW % 4 == 0: a quad is inside the image or outside it
        v[i] = *reinterpret_cast<const f32x4_t*>(s);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) if (4 * q + e < np) v[i][e] = s[e];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = tid + i * 256, c = t / PQ, q = t % PQ;
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[c * ROW + 4 * q + e] = v[i][e];
  }
  __syncthreads();
  const int ny = min(CT, a.c_pad - c0);   // channels written, zero padding included
#pragma unroll
  for (int i = 0; i < CPP * PT / 256; ++i) {
    const int t = tid + i * 256, p = t / CPP, cc = (t % CPP) * EPC;
    if (p >= np || cc >= ny) continue;
    T o[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e) o[e] = Elt<T>::from_f(tile[(cc + e) * ROW + p]);
    T* d = y + (int64_t)p * a.c_pad + cc;
    if (a.vec_c) {   // c_pad is a multiple of the chunk
      *reinterpret_cast<u32x4_t*>(d) = *reinterpret_cast<const u32x4_t*>(o);
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) if (cc + e < ny) d[e] = o[e];
    }
  }
}

template <typename T, int CT>
__device__ __forceinline__ void unpack_body(const vrs_pack_args& a) {
  constexpr int PT = 4096 / CT, ROW = PT + 1, PQ = PT / 4;
  constexpr int EPC = 16 / (int)sizeof(T), CPP = CT / EPC, NL = CPP * PT / 256;
  __shared__ float tile[CT * ROW];
  int b, c0;
  int64_t p0;
  if (!layout_tile<T, CT>(a, b, c0, p0)) return;
  const T* x = reinterpret_cast<const T*>(a.x) + ((int64_t)b * a.HW + p0) * a.c_pad + c0;
  float* y = reinterpret_cast<float*>(a.y) + ((int64_t)b * a.C + c0) * a.HW + p0;
  const int np = (int)min((int64_t)PT, a.HW - p0), nc = min(CT, a.C - c0);
  const int tid = threadIdx.x;
  T v[NL][EPC];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int t = tid + i * 256, p = t / CPP, cc = (t % CPP) * EPC;
    if (p >= np || cc >= nc) continue;
    const T* s = x + (int64_t)p * a.c_pad + cc;
    if (a.vec_c) {   // the chunk stays inside the pixel's row (pitch a multiple of it)
      *reinterpret_cast<u32x4_t*>(v[i]) = *reinterpret_cast<const u32x4_t*>(s);
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) if (cc + e < nc) v[i][e] = s[e];
    }
  }
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int t = tid + i * 256, p = t / CPP, cc = (t % CPP) * EPC;
    if (p >= np || cc >= nc) continue;
#pragma unroll
    for (int e = 0; e < EPC; ++e) tile[(cc + e) * ROW + p] = Elt<T>::to_f(v[i][e]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = tid + i * 256, c = t / PQ, q = t % PQ;
    if (c >= nc || 4 * q >= np) continue;
    float* d = y + (int64_t)c * a.HW + 4 * q;
    const float* s = &tile[c * ROW + 4 * q];
    if (a.vec_p) {
      *reinterpret_cast<f32x4_t*>(d) = (f32x4_t){s[0], s[1], s[2], s[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) if (4 * q + e < np) d[e] = s[e];
    }
  }
}

}  // namespace

#define VRS_LAYOUT(DT, T, CT)                                                                                      \
  extern "C" __global__ __launch_bounds__(256) void vrs_pack_nchw_##DT##_c##CT(vrs_pack_args a) {                 \
    pack_body<T, CT>(a);                                                                                           \
  }                                                                                                                \
  extern "C" __global__ __launch_bounds__(256) void vrs_unpack_nchw_##DT##_c##CT(vrs_pack_args a) {               \
    unpack_body<T, CT>(a);                                                                                         \
  }
// vrs_[un]pack_nchw_<type>_c<channels per tile>
VRS_LAYOUT(bf16, bf16_t, 8)
VRS_LAYOUT(bf16, bf16_t, 64)
VRS_LAYOUT(f32, float, 8)
VRS_LAYOUT(f32, float, 64)
