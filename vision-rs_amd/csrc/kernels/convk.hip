// Split-K implicit-GEMM conv for small problems (gfx950): batch-1 and
// batch-few layers, whose 64x64 and larger tiles leave most of the 256 CUs
// without a workgroup while each busy one walks the whole K range.
//
// Semantics as conv_body.h: y = act(scale * conv(x, w) + shift) + res, folded
// BN, k up to 5, any stride, optional fused nearest-2x upsample, NHWC or flat
// (channel-major float32) output; bf16 and float32 with Cin % 8 == 0, or e4m3
// weights and activations (element type uint8_t) with Cin % 64 == 0, whose
// output and residual are bf16 or e4m3.
//
// Latency bounds these layers, not bytes or flops: the time is the chain of
// dependent waits of one workgroup.  So the output tile is one MFMA tile (32
// channels x 32 pixels, or 16 x 16), four to sixteen times the workgroups of
// the 64x64 tile, and the KW waves of a workgroup share its K range: wave w
// takes the 128-byte steps w, w + KW, ... of every row.  A wave stages its own
// steps: global loads of whole 128-byte row pieces (eight lanes a row; loading
// MFMA fragments directly, a row per lane, was bound by the 64 lines each load
// touches), three steps in flight in registers, through LDS rows that no
// other wave touches, so the loop has no barrier.  At the end the KW partial
// tiles are summed through LDS in a fixed order (the result does not depend on
// timing).  KW = 1 (short K): four waves take four neighbouring
// pixel tiles and nothing is summed.
// Measured (graph launches, of which an empty one takes about 3.5 us), best
// earlier tile -> this kernel: float32 3x3 128->128 at 40x40 x 1 58 -> 11.7 us
// (MFMA floor 3.4), 3x3 512->64 at 20x20 x 1 214 -> 12.4 us, 1x1 256->256 at
// 20x20 x 1 17.1 -> 4.9 us, 3x3 32->32 at 40x40 x 4 18.5 -> 6.7 us; bfloat16
// 3x3 512->64 at 20x20 x 1 23.6 -> 7.0 us, 3x3 128->128 at 20x20 x 1 8.5 ->
// 4.8 us, 3x3/s2 512->512 at 40x40 x 1 24.7 -> 11.4 us, 1x1 384->256 at 20x20
// x 1 5.2 -> 4.4 us.
#include "common.h"

namespace {

// One K slice of a TS x TS tile.
template <typename T, int TS> struct Unit;
template <> struct Unit<bf16_t, 32> {
  using acc_t = f32x16_t;
  static __device__ __forceinline__ acc_t mma(u32x4_t a, u32x4_t b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
};
template <> struct Unit<bf16_t, 16> {
  using acc_t = f32x4_t;
  static __device__ __forceinline__ acc_t mma(u32x4_t a, u32x4_t b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
};
// float32: step j takes element j of every lane's four
template <> struct Unit<float, 32> {
  using acc_t = f32x16_t;
  static __device__ __forceinline__ acc_t mma(u32x4_t a, u32x4_t b, acc_t c) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[j]), __uint_as_float(b[j]), c, 0, 0, 0);
    return c;
  }
};
template <> struct Unit<float, 16> {
  using acc_t = f32x4_t;
  static __device__ __forceinline__ acc_t mma(u32x4_t a, u32x4_t b, acc_t c) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[j]), __uint_as_float(b[j]), c, 0, 0, 0);
    return c;
  }
};

// e4m3: 32 bytes of k per lane, unit block scales
template <> struct Unit<uint8_t, 32> {
  using acc_t = f32x16_t;
  static __device__ __forceinline__ acc_t mma(const i32x8_t& a, const i32x8_t& b, acc_t c) { return mfma32_fp8_k64(a, b, c); }
};
template <> struct Unit<uint8_t, 16> {
  using acc_t = f32x4_t;
  static __device__ __forceinline__ acc_t mma(const i32x8_t& a, const i32x8_t& b, acc_t c) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
  }
};

// ALIGNED: a tap's channels are whole steps (128 bytes of a row), so the tap
// of a step is the same for all lanes; otherwise each lane follows its own
// 16-byte chunk (which never straddles two taps: Cin % 8 == 0).
template <typename T, int TS, int KW, int NT, bool ALIGNED>
__device__ __forceinline__ void convk_body(const vrs_convk_args& k) {
  const vrs_conv_args& a = k.c;
  using acc_t = typename Unit<T, TS>::acc_t;
  constexpr int ES = (int)sizeof(T), U = 16 / ES;    // elements per 16-byte chunk
  constexpr int CPS = 8;                              // chunks per row and step
  constexpr int NG = 64 / TS;                         // lane groups along K of one MFMA
  constexpr int RL = TS / 8;                          // loads per lane, operand and step (8 rows of 128 B each)
  constexpr int DEPTH = 3;             // steps in flight
  constexpr int ROW = 128 + 16;                       // LDS row: 128 bytes and a pad against bank conflicts
  constexpr int NQ = TS == 32 ? 4 : 1;                // accumulator quads per lane
  static_assert(KW == 1 || NT == 1, "one shared tile, or one tile per wave");
  __shared__ __attribute__((aligned(16))) unsigned char lds[KW * NT][2 * TS * ROW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* const sa = lds[wave];
  unsigned char* const sb = sa + TS * ROW;

  // k.chan_major: workgroups of one channel tile are neighbours (an XCD then
  // holds few weight rows and all pixels), else those of one pixel tile
  const int logical = xcd_remap(blockIdx.x, gridDim.x);
  const int minor = k.chan_major ? a.tiles_n : a.tiles_m;
  const int q = logical / minor, r = logical - q * minor;
  const int m0 = (k.chan_major ? q : r) * TS;
  const int n0 = ((k.chan_major ? r : q) * NT + (KW == 1 ? wave : 0)) * TS;

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w, a.w_bytes);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.x_bytes);
  const __amdgpu_buffer_rsrc_t rx2 = make_rsrc(a.x2, a.c_split ? a.x2_bytes : 0);
  const int HWo = a.Ho * a.Wo;
  const float inv_hwo = 1.0f / (float)HWo, inv_wo = 1.0f / (float)a.Wo;

  // staging: lane takes chunk (lane & 7) of rows (lane >> 3) + 8 i of both operands
  const int ch = lane & 7, r0 = lane >> 3;
  uint32_t a_off[RL], b_off[RL], b_off2[ALIGNED ? RL : 1], taps[RL];
#pragma unroll
  for (int i = 0; i < RL; ++i) {
    const int co = m0 + r0 + 8 * i, m = n0 + r0 + 8 * i;
    a_off[i] = co < a.Cout ? (uint32_t)co * (uint32_t)(a.K * ES) + ch * 16u : kOOB;
    const bool ok = m < a.M;
    int rr, ox;
    const int bb = fdivmod(ok ? m : 0, HWo, inv_hwo, rr);
    const int oy = fdivmod(rr, a.Wo, inv_wo, ox);
    const int iy0 = oy * a.stride - a.pad, ix0 = ox * a.stride - a.pad;
    b_off[i] = (uint32_t)((((int64_t)bb * a.H + iy0) * a.W + ix0) * a.x_pitch) * (uint32_t)ES + (ALIGNED ? ch * 16u : 0u);
    if constexpr (ALIGNED)
      b_off2[i] = ok ? (uint32_t)((((int64_t)bb * a.H2 + (oy >> 1)) * a.W2 + (ox >> 1)) * a.x2_pitch) * (uint32_t)ES +
                           ch * 16u
                     : kOOB;
    // the taps of this pixel that lie inside the image, a bit each (k <= 5)
    uint32_t cols = 0;
    for (int kx = 0; kx < a.kw; ++kx) cols |= (unsigned)(ix0 + kx) < (unsigned)a.W ? 1u << kx : 0u;
    taps[i] = 0;
    for (int ky = 0; ky < a.kh; ++ky)
      if ((unsigned)(iy0 + ky) < (unsigned)a.H) taps[i] |= cols << (ky * a.kw);
    if (!ok) taps[i] = 0;
  }

  // steps wave, wave + KW, ...; K is gpr 16-byte chunks per row, k.gpt per tap
  const int gpr = a.K / U;
  const int steps = (gpr + CPS - 1) / CPS;
  const int first = KW == 1 ? 0 : wave;
  const int n = (steps - first + KW - 1) / KW;
  int g = first * CPS;                                // next step's first chunk
  const float inv_gpt = 1.0f / (float)k.gpt;
  int t_c = 0, t_tap = 0;                             // ALIGNED: its tap and chunk inside the tap
  if (ALIGNED) {
    t_tap = g / k.gpt;
    t_c = g - t_tap * k.gpt;
  }
  u32x4_t va[DEPTH][RL], vb[DEPTH][RL];
  auto load = [&](u32x4_t (&wa)[RL], u32x4_t (&wb)[RL]) {
    // chunks past K (the last step's tail, steps past the last): zeros, at tap 0
    // (the look-ahead's own tap may be one of no filter)
    uint32_t dead = g < gpr ? 0u : kOOB;
    int tap = g < gpr ? t_tap : 0, c = t_c;
    if constexpr (!ALIGNED) {
      const int gl = g + ch;
      dead = gl < gpr ? 0u : kOOB;
      tap = fdivmod(gl < gpr ? gl : 0, k.gpt, inv_gpt, c);
    }
    const int ky = tap * k.inv_kw >> 8, kx = tap - ky * a.kw;
    const uint32_t off = (uint32_t)((ky * a.W + kx) * a.x_pitch) * (uint32_t)ES + c * 16u;
#pragma unroll
    for (int i = 0; i < RL; ++i) wa[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, (a_off[i] + g * 16u) | dead, 0, 0);
    const bool lo = ALIGNED && c * U < a.c_split;     // uniform; 1x1 conv: the half-size source
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const uint32_t in = (taps[i] >> tap & 1u) ? b_off[i] + off : kOOB;
      if constexpr (ALIGNED)
        wb[i] = __builtin_amdgcn_raw_buffer_load_b128(lo ? rx2 : rx, (lo ? b_off2[i] + c * 16u : in) | dead, 0, 0);
      else
        wb[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, in | dead, 0, 0);
    }
    g += KW * CPS;
    if constexpr (ALIGNED) {
      t_c += k.d_chunk;
      t_tap += k.d_tap;
      if (t_c >= k.gpt) { t_c -= k.gpt; ++t_tap; }
    }
  };
  acc_t acc;
#pragma unroll
  for (int e = 0; e < NQ * 4; ++e) acc[e] = 0.f;
  constexpr int FB = ES == 1 ? 32 : 16;               // bytes of a row per lane and slice
  const int f_off = (lane % TS) * ROW + (lane / TS) * FB;
  // one step: the staged rows through this wave's own LDS (LDS operations of
  // one wave are in order: no barrier) into MFMA fragments.  The wave barriers
  // are for the compiler, which sees only each lane's own addresses: they keep
  // the stores before the fragment reads and these before the next step's stores.
  auto step = [&](const u32x4_t (&wa)[RL], const u32x4_t (&wb)[RL]) {
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      *reinterpret_cast<u32x4_t*>(sa + (r0 + 8 * i) * ROW + ch * 16) = wa[i];
      *reinterpret_cast<u32x4_t*>(sb + (r0 + 8 * i) * ROW + ch * 16) = wb[i];
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto mma = [&]() {
    if constexpr (ES == 1) {
      constexpr int NS = 128 / (NG * FB);
      i32x8_t fa[NS], fb[NS];
      auto ld32 = [&](const unsigned char* p) {
        const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(p), hi = *reinterpret_cast<const u32x4_t*>(p + 16);
        return (i32x8_t){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      };
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        fa[s] = ld32(sa + f_off + s * NG * FB);
        fb[s] = ld32(sb + f_off + s * NG * FB);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s = 0; s < NS; ++s) acc = Unit<T, TS>::mma(fa[s], fb[s], acc);
    } else {
      u32x4_t fa[CPS / NG], fb[CPS / NG];
#pragma unroll
      for (int s = 0; s < CPS / NG; ++s) {
        fa[s] = *reinterpret_cast<const u32x4_t*>(sa + f_off + s * NG * 16);
        fb[s] = *reinterpret_cast<const u32x4_t*>(sb + f_off + s * NG * 16);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s = 0; s < CPS / NG; ++s) acc = Unit<T, TS>::mma(fa[s], fb[s], acc);
    }
  };

#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(va[d], vb[d]);

  // this thread's output quads: channels m0 + qd * 8 + hq ..+3 of its lane's
  // pixel; with KW > 1 thread t finishes quad t.  Their constants arrive under
  // the K loop.
  const int hq = TS == 32 ? (lane >> 5) * 4 : (lane >> 4) * 4;
  const int qd0 = KW == 1 ? 0 : (TS == 32 ? tid >> 6 : 0);
  float sc[KW == 1 ? NQ : 1][4], sh[KW == 1 ? NQ : 1][4];
  const bool finishes = KW == 1 || tid < 64 * NQ;
  const int m = n0 + lane % TS;
  int rr;
  const int bb = fdivmod(m < a.M ? m : 0, HWo, inv_hwo, rr);
  if (finishes) {
#pragma unroll
    for (int i = 0; i < (KW == 1 ? NQ : 1); ++i) {
      const int co = m0 + (qd0 + i) * 8 + hq;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int cc = min(co + e, a.Cout - 1);
        sc[i][e] = a.scale[cc];
        sh[i][e] = a.shift[cc];
      }
    }
  }

  for (int i = 0; i < n;) {   // DEPTH steps per turn, left after the last one
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      step(va[d], vb[d]);
      load(va[d], vb[d]);
      mma();
      if (++i >= n) break;
    }
  }

  auto finish = [&](const f32x4_t& s, int qd, const float (&qs)[4], const float (&qt)[4]) {
    const int co = m0 + qd * 8 + hq;
    if (m >= a.M || co >= a.Cout) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = s[e] * qs[e] + qt[e];
      if (a.act == VRS_ACT_SILU) v[e] = silu_t<T>(v[e]);
    }
    if (a.res) {   // NHWC views: whole aligned quads (host)
      const int64_t ro = bb * a.r_sb + rr * a.r_sp + co;
      if (ES == 1 && a.res_f8) {
        float d[4];
        fp8x4_to_f32(*reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.res) + ro), a.res_step, d);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += d[e];
      } else if constexpr (ES <= 2) {
        const u32x2_t rv = *reinterpret_cast<const u32x2_t*>(static_cast<const bf16_t*>(a.res) + ro);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += __uint_as_float((e & 1) ? (rv[e >> 1] & 0xffff0000u) : (rv[e >> 1] << 16));
      } else {
        const f32x4_t rv = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(a.res) + ro);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += rv[e];
      }
    }
    const int64_t yo = bb * a.y_sb + rr * a.y_sp + (int64_t)co * a.y_sc;
    if (a.y_f32) {
      float* yp = reinterpret_cast<float*>(a.y) + yo;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (co + e < a.Cout) yp[e * a.y_sc] = v[e];
    } else if constexpr (ES <= 2) {
      const u32x2_t h = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      if (ES == 1 && a.out_step > 0.f) {   // e4m3 of the bf16 value
        uint32_t lim = __float_as_uint(448.f * a.out_step) >> 16;
        lim |= lim << 16;
        *reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(a.y) + yo) =
            bf16x2_to_fp8x2(h[0], lim, a.out_step) | (bf16x2_to_fp8x2(h[1], lim, a.out_step) << 16);
      } else {
        *reinterpret_cast<u32x2_t*>(static_cast<bf16_t*>(a.y) + yo) = h;
      }
    } else {
      *reinterpret_cast<f32x4_t*>(reinterpret_cast<T*>(a.y) + yo) = (f32x4_t){v[0], v[1], v[2], v[3]};
    }
  };

  if constexpr (KW == 1) {
#pragma unroll
    for (int i = 0; i < NQ; ++i)
      finish((f32x4_t){acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]}, i, sc[i], sh[i]);
  } else {
    // each wave's partial tile over its own staging rows, summed in a fixed order
    static_assert(NQ * 64 * 16 <= 2 * TS * ROW, "partial tile fits the staging rows");
    f32x4_t* part = reinterpret_cast<f32x4_t*>(sa);
#pragma unroll
    for (int i = 0; i < NQ; ++i)
      part[i * 64 + lane] = (f32x4_t){acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]};
    __syncthreads();
    if (finishes) {
      // pairwise: half the rounding steps of a running sum
      f32x4_t s[KW];
#pragma unroll
      for (int w = 0; w < KW; ++w) s[w] = reinterpret_cast<const f32x4_t*>(lds[w])[tid];
#pragma unroll
      for (int d = 1; d < KW; d *= 2)
#pragma unroll
        for (int w = 0; w + d < KW; w += 2 * d) s[w] += s[w + d];
      finish(s[0], qd0, sc[0], sh[0]);
    }
  }
}

// waves per SIMD to leave registers for: three staged steps of a 32x32 tile
// take 96 of them and spill at four waves
constexpr int convk_waves(int ts, int kw) { return ts == 16 ? 4 : kw == 8 ? 2 : 3; }

}  // namespace

#define VRS_CONVK(DT, T, TS, KW, NT)                                                                               \
  extern "C" __global__ __launch_bounds__(64 * KW * NT, convk_waves(TS, KW)) void vrs_conv_##DT##_s##TS##_w##KW##_a(vrs_convk_args a) { \
    convk_body<T, TS, KW, NT, true>(a);                                                                             \
  }                                                                                                                 \
  extern "C" __global__ __launch_bounds__(64 * KW * NT, convk_waves(TS, KW)) void vrs_conv_##DT##_s##TS##_w##KW##_g(vrs_convk_args a) { \
    convk_body<T, TS, KW, NT, false>(a);                                                                            \
  }
#define VRS_CONVK_TYPE(DT, T)  \
  VRS_CONVK(DT, T, 32, 4, 1)   \
  VRS_CONVK(DT, T, 32, 8, 1)   \
  VRS_CONVK(DT, T, 16, 1, 4)   \
  VRS_CONVK(DT, T, 16, 4, 1)   \
  VRS_CONVK(DT, T, 16, 8, 1)
// vrs_conv_<type>_s<tile>_w<waves sharing K>_<a: taps of whole steps, g: any Cin % 8 == 0>
VRS_CONVK_TYPE(bf16, bf16_t)
VRS_CONVK_TYPE(f32, float)
VRS_CONVK_TYPE(fp8, uint8_t)
