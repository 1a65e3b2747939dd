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
// Small maps (SMALL): a tile takes several whole images, else most of its lanes
// would have no pixel: 65536 maps of 3 channels at 1x1 65 -> 3.8 us, of 512
// channels 580 -> 41 us; 16384 of 64 channels at 3x3 32 -> 16 us.
#include "common.h"

namespace {

// The tile of this workgroup: channels from c0, pixels from p0 of image b.
// SMALL: a.imgs whole images from b, whose NHWC rows follow each other.
template <int CT, bool SMALL>
__device__ __forceinline__ bool layout_tile(const vrs_pack_args& a, int& b, int& c0, int64_t& p0) {
  constexpr int PT = 4096 / CT;
  const uint32_t logical = a.first + (uint32_t)xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t r = logical / (uint32_t)a.tiles_c;
  c0 = (int)(logical - r * (uint32_t)a.tiles_c) * CT;
  const uint32_t g = SMALL ? r : r / (uint32_t)a.tiles_p;
  b = (int)(SMALL ? g * (uint32_t)a.imgs : g);
  p0 = SMALL ? 0 : (int64_t)(r - g * (uint32_t)a.tiles_p) * PT;
  return b < a.N;
}

// SMALL: the float32 side of a tile is one run of nc * HW values per image.
// Value t of them all: its offset from the first image's run and its place in
// the LDS tile.
struct layout_runs {
  int hw, run, total;
  float inv_hw, inv_run;
  __device__ layout_runs(const vrs_pack_args& a, int imgs, int nc)
      : hw((int)a.HW), run(nc * (int)a.HW), total(imgs * nc * (int)a.HW), inv_hw(1.0f / (float)hw),
        inv_run(1.0f / (float)run) {}
  __device__ int64_t at(const vrs_pack_args& a, int t, int row, int& lds) const {
    int r, p;
    const int j = fdivmod(t, run, inv_run, r), c = fdivmod(r, hw, inv_hw, p);
    lds = c * row + j * hw + p;
    return (int64_t)j * a.C * hw + r;
  }
};

template <typename T, int CT, bool SMALL>
__device__ __forceinline__ void pack_body(const vrs_pack_args& a) {
  constexpr int PT = 4096 / CT, ROW = PT + 1, PQ = PT / 4;
  constexpr int EPC = 16 / (int)sizeof(T), CPP = CT / EPC;   // elements per chunk, chunks per pixel
  __shared__ float tile[CT * ROW];
  int b, c0;
  int64_t p0;
  if (!layout_tile<CT, SMALL>(a, b, c0, p0)) return;
  const float* x = reinterpret_cast<const float*>(a.x) + ((int64_t)b * a.C + c0) * a.HW + p0;
  T* y = reinterpret_cast<T*>(a.y) + ((int64_t)b * a.HW + p0) * a.c_pad + c0;
  const int imgs = SMALL ? min(a.imgs, a.N - b) : 1;
  // valid pixels and (may be <= 0) channels
  const int np = SMALL ? imgs * (int)a.HW : (int)min((int64_t)PT, a.HW - p0), nc = min(CT, a.C - c0);
  const int tid = threadIdx.x;
  if constexpr (SMALL) {
    if (nc > 0) {
      const layout_runs runs(a, imgs, nc);
      float v[16];
      int at[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = tid + i * 256;
        if (t < runs.total) v[i] = x[runs.at(a, t, ROW, at[i])];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (tid + i * 256 < runs.total) tile[at[i]] = v[i];
    }
  } else {
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
  }
  __syncthreads();
  const int ny = min(CT, a.c_pad - c0);   // channels written, zero padding included
#pragma unroll
  for (int i = 0; i < CPP * PT / 256; ++i) {
    const int t = tid + i * 256, p = t / CPP, cc = (t % CPP) * EPC;
    if (p >= np || cc >= ny) continue;
    T o[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e)
      o[e] = Elt<T>::from_f(!SMALL || cc + e < nc ? tile[(cc + e) * ROW + p] : 0.f);   // (SMALL: only nc rows are filled)
    T* d = y + (int64_t)p * a.c_pad + cc;
    if (a.vec_c) {   // c_pad is a multiple of the chunk
      *reinterpret_cast<u32x4_t*>(d) = *reinterpret_cast<const u32x4_t*>(o);
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) if (cc + e < ny) d[e] = o[e];
    }
  }
}

template <typename T, int CT, bool SMALL>
__device__ __forceinline__ void unpack_body(const vrs_pack_args& a) {
  constexpr int PT = 4096 / CT, ROW = PT + 1, PQ = PT / 4;
  constexpr int EPC = 16 / (int)sizeof(T), CPP = CT / EPC, NL = CPP * PT / 256;
  __shared__ float tile[CT * ROW];
  int b, c0;
  int64_t p0;
  if (!layout_tile<CT, SMALL>(a, b, c0, p0)) return;
  const T* x = reinterpret_cast<const T*>(a.x) + ((int64_t)b * a.HW + p0) * a.c_pad + c0;
  float* y = reinterpret_cast<float*>(a.y) + ((int64_t)b * a.C + c0) * a.HW + p0;
  const int imgs = SMALL ? min(a.imgs, a.N - b) : 1;
  const int np = SMALL ? imgs * (int)a.HW : (int)min((int64_t)PT, a.HW - p0), nc = min(CT, a.C - c0);
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
  if constexpr (SMALL) {
    const layout_runs runs(a, imgs, nc);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = tid + i * 256;
      int at;
      if (t < runs.total) {
        const int64_t d = runs.at(a, t, ROW, at);
        y[d] = tile[at];
      }
    }
  } else {
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
}

}  // namespace

#define VRS_LAYOUT(DT, T, CT, TAG, SMALL)                                                                          \
  extern "C" __global__ __launch_bounds__(256) void vrs_pack_nchw_##DT##_##TAG##CT(vrs_pack_args a) {             \
    pack_body<T, CT, SMALL>(a);                                                                                    \
  }                                                                                                                \
  extern "C" __global__ __launch_bounds__(256) void vrs_unpack_nchw_##DT##_##TAG##CT(vrs_pack_args a) {           \
    unpack_body<T, CT, SMALL>(a);                                                                                  \
  }
// vrs_[un]pack_nchw_<type>_<c: tiles of one image, i: of whole images><channels per tile>
VRS_LAYOUT(bf16, bf16_t, 8, c, false)
VRS_LAYOUT(bf16, bf16_t, 64, c, false)
VRS_LAYOUT(f32, float, 8, c, false)
VRS_LAYOUT(f32, float, 64, c, false)
VRS_LAYOUT(bf16, bf16_t, 8, i, true)
VRS_LAYOUT(bf16, bf16_t, 64, i, true)
VRS_LAYOUT(f32, float, 8, i, true)
VRS_LAYOUT(f32, float, 64, i, true)
