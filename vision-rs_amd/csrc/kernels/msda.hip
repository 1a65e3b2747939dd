// Multi-scale deformable attention (RF-DETR decoder cross-attention) for gfx950.
// There is no reference function (the reference has no deformable attention);
// the semantics are the published Deformable-DETR formulation that BASELINE
// config 4 names: for each (b, q, head)
//   out[d] = sum_{l,p} attw[l,p] * bilinear(V_l[:, :, head, d],
//                                           x = (ref_x + off_x) * W_l - 0.5,
//                                           y = (ref_y + off_y) * H_l - 0.5)
// with zero padding outside the map (grid_sample bilinear, zeros,
// align_corners=False).
//
// Gather-bound.  The value tensor [B, S, heads, 32] keeps each (pixel, head)
// row of 32 floats (128 bytes) contiguous; 8 lanes own one head and fetch a
// corner row as 8 x 16-byte loads, so one wave64 serves all 8 heads of one
// query and every corner fetch is a full 128-byte segment per head.  The
// point loop is unrolled at compile time (P <= 4) and each level has a wave of
// its own, so all corner fetches of a query are independent loads in flight
// together; sampling locations and weights are read once per lane group with
// 8-byte / 4-byte loads.
#include "common.h"

namespace {

// Sampling coordinate (ref + off) * size - 0.5 as a rounded add, a rounded
// multiply and a rounded subtract -- no fused multiply-add -- so every
// bilinear corner and weight is the one the float32 CPU restatement (built
// with contraction off) computes; a contracted form moves a coordinate by up
// to half an ulp (~4e-6 at the 80-wide level), which shows in the outputs at
// the 1e-4 parity bar.
__device__ __forceinline__ float sample_coord(float r, float o, int n) {
#pragma clang fp contract(off)
  const float loc = r + o;
  const float scaled = loc * (float)n;
  return scaled - 0.5f;
}

// Any number of points: runtime loops (what the unrolled kernels do not cover).
__device__ __forceinline__ void msda_any(const vrs_msda_args& a) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int part = (int)(gid & 7);
  const int64_t bqh = gid >> 3;
  if (bqh >= (int64_t)a.B * a.Q * a.heads) return;
  const int h = (int)(bqh % a.heads);
  const int64_t bq = bqh / a.heads;
  const int b = (int)(bq / a.Q);
  const float rx = a.ref[bq * 2 + 0], ry = a.ref[bq * 2 + 1];
  const int64_t row = (int64_t)a.heads * 32;
  const float* vb = a.value + (int64_t)b * a.S * row + h * 32 + part * 4;
  const int64_t obase = bqh * a.L * a.P;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int l = 0; l < a.L; ++l) {
    const int Hl = a.lh[l], Wl = a.lw[l];
    const float* vl = vb + (int64_t)a.lstart[l] * row;
    for (int p = 0; p < a.P; ++p) {
      const int64_t oi = obase + l * a.P + p;
      const float ix = sample_coord(rx, a.off[2 * oi], Wl);
      const float iy = sample_coord(ry, a.off[2 * oi + 1], Hl);
      const float w = a.attw[oi];
      const float fx = floorf(ix), fy = floorf(iy);
      const int x0 = (int)fx, y0 = (int)fy;
      const float ax1 = ix - fx, ay1 = iy - fy;
      const float ax0 = 1.f - ax1, ay0 = 1.f - ay1;
      const int xs[2] = {x0, x0 + 1}, ys[2] = {y0, y0 + 1};
      const float wx[2] = {ax0, ax1}, wy[2] = {ay0, ay1};
      for (int cy = 0; cy < 2; ++cy)
        for (int cx = 0; cx < 2; ++cx) {
          if ((unsigned)xs[cx] >= (unsigned)Wl || (unsigned)ys[cy] >= (unsigned)Hl) continue;
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(vl + ((int64_t)ys[cy] * Wl + xs[cx]) * row);
          acc += (w * wy[cy] * wx[cx]) * v;
        }
    }
  }
  *reinterpret_cast<f32x4_t*>(a.out + bq * row + h * 32 + part * 4) = acc;
}

// P points, L <= 8 levels, split by level: a workgroup takes eight consecutive
// (query, head) rows of one image -- a query at eight heads -- and its wave l
// level l, so the rows' corner fetches spread over L waves, each lane with its
// 4 P independent loads in flight; the partial sums meet in LDS.  The general
// kernel's runtime loops wait for a point's offsets before the next point's
// are asked for, 2 L P dependent round trips; here there are two.  Corners come
// by buffer loads (32-bit offsets from the image, zero outside), which take no
// branch and half the address registers.
// Workgroups are dealt round-robin over the 8 XCDs; the XCD-aware order gives
// each XCD a contiguous run of queries -- whole images at B*Q/8 queries per
// XCD -- so the corner rows one image's queries share are fetched into one
// L2 rather than into all eight.
// The gather's latency and HBM bound it.  Measured at 8 heads, calls back to
// back (general kernel -> this one): 8 x 300 queries on 80x80, 3 levels x 4
// points 23.5 -> 9.2 us, 4 x 2 16.7 -> 6.8; 16 x 900 on 120x120, 3 x 4 91 -> 55
// us (6.2 TB/s on the bytes read and written once).  With 64-bit addresses and
// branches around the corners, 4 x 4: 11.5 -> 11.1 us (8 x 300), 66.5 -> 64.6.
template <int P>
__device__ __forceinline__ void msda_split_body(const vrs_msda_args& a) {
  __shared__ f32x4_t part[8][64];
  const int lane = threadIdx.x & 63, l = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t rows = (uint32_t)a.Q * (uint32_t)a.heads, per = (rows + 7) / 8;   // of one image (host: < 2^31)
  const uint32_t logical = (uint32_t)xcd_remap(blockIdx.x, gridDim.x), b = logical / per;
  const uint32_t r = (logical - b * per) * 8 + (lane >> 3);
  const uint32_t pc = lane & 7;   // 4-channel part
  const bool live = r < rows;
  const int64_t bqh = (int64_t)b * rows + r;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (live) {
    const uint32_t q = r / (uint32_t)a.heads, h = r - q * (uint32_t)a.heads;
    const float2 ref = {a.ref[((int64_t)b * a.Q + q) * 2], a.ref[((int64_t)b * a.Q + q) * 2 + 1]};
    const int64_t row = (int64_t)a.heads * 32;
    const uint32_t px = (uint32_t)row * 4;   // bytes of a pixel (host: an image < 2^31)
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.value + (int64_t)b * a.S * row, (int64_t)a.S * row * 4);
    const int Hl = a.lh[l], Wl = a.lw[l];
    const uint32_t base = (uint32_t)a.lstart[l] * px + h * 128u + pc * 16u;
    const float* offs = a.off + (bqh * a.L + l) * (2 * P);
    const float* attw = a.attw + (bqh * a.L + l) * P;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const float2 off = *reinterpret_cast<const float2*>(offs + 2 * p);
      const float w = attw[p];
      const float ix = sample_coord(ref.x, off.x, Wl);
      const float iy = sample_coord(ref.y, off.y, Hl);
      const float fx = floorf(ix), fy = floorf(iy);
      const int x0 = (int)fx, y0 = (int)fy;
      const float ax1 = ix - fx, ay1 = iy - fy;
      const float wx[2] = {1.f - ax1, ax1}, wy[2] = {w * (1.f - ay1), w * ay1};
      const uint32_t o = base + ((uint32_t)y0 * (uint32_t)Wl + (uint32_t)x0) * px;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int dx = c & 1, dy = c >> 1;
        // a corner outside the map takes weight 0 and value 0: nothing, also
        // where a coordinate or the weight is not finite
        const bool in = (uint32_t)x0 + dx < (uint32_t)Wl && (uint32_t)y0 + dy < (uint32_t)Hl;
        const f32x4_t v = __builtin_bit_cast(
            f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, in ? o + (dy * (uint32_t)Wl + dx) * px : kOOB, 0, 0));
        acc += (in ? wy[dy] * wx[dx] : 0.f) * v;
      }
    }
  }
  part[l][lane] = acc;
  __syncthreads();
  if (l == 0 && live) {
    f32x4_t sum = part[0][lane];
    for (int i = 1; i < a.L; ++i) sum += part[i][lane];
    *reinterpret_cast<f32x4_t*>(a.out + bqh * 32 + pc * 4) = sum;
  }
}

}  // namespace

extern "C" __global__ __launch_bounds__(512) void vrs_msda_p1_f32(vrs_msda_args a) { msda_split_body<1>(a); }
extern "C" __global__ __launch_bounds__(512) void vrs_msda_p2_f32(vrs_msda_args a) { msda_split_body<2>(a); }
extern "C" __global__ __launch_bounds__(512) void vrs_msda_p3_f32(vrs_msda_args a) { msda_split_body<3>(a); }
extern "C" __global__ __launch_bounds__(512) void vrs_msda_p4_f32(vrs_msda_args a) { msda_split_body<4>(a); }
extern "C" __global__ __launch_bounds__(256) void vrs_msda_f32(vrs_msda_args a) { msda_any(a); }
