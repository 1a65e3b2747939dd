// Detect-head post-processing on gfx950.
//
// Stage 1: LTRB -> xywh decode, sigmoid per class, argmax, threshold -- the
// host loops of examples/yolo26.rs:1488-1528 with the anchor grid of
// loss/anchor.rs:47-66.  The argmax follows Rust's Iterator::max_by with
// partial_cmp().unwrap_or(Equal): the running best is kept only if it compares
// Greater, so the last of equal maxima wins and a NaN compares Equal.  A kept
// anchor gets the unique 64-bit key (score_bits << 32) | (0xffffffff -
// anchor): ordering keys descending is the stable descending sort of
// examples/yolo26.rs:1529 (equal scores keep ascending anchor order); sigmoid
// scores are non-negative so their IEEE bits order like the values.
//
// Stage 2 (one workgroup per image): exact top-k (k = min(count, max_det)).
// With at most TOPK_MAX kept anchors every key is gathered into LDS and
// bitonic-sorted.  Otherwise a most-significant-digit radix select raises a
// threshold 11 bits at a time and stops as soon as the keys at or above it
// fit the LDS buffer (at the latest after the 6th digit, when the threshold
// is the k-th largest key itself); those keys are gathered and sorted.
#include "common.h"

// four floats at any dword address (the workspace's boxes start after 8-byte keys)
typedef float f32x4_any __attribute__((vector_size(16), aligned(4)));

// Stage 1 reads the logits once (bs64 640, 80 classes: 172 MB); with a sigmoid
// per logit and a load waited for at a time it took 61 us.  Only the largest
// logit's sigmoid is computed: the sigmoid's rounding (a few ulp) can only
// reorder logits within 2e-5 of each other when they are negative (its relative
// slope is at least 1/2 there: 80 ulp), within 1e-3 up to 5 (at least 1/150: 50
// ulp), any at or above 5, where it flattens to 1, and any below -80, where it
// underflows.  An anchor whose second largest logit is that near, or that has
// a NaN, goes through the classes again in order (those near enough; all of
// them for NaN and underflow), so the class and score are those of the plain
// loop, bit for bit.  One anchor per
// thread, eight classes in flight: 34.3 us = 5.2 TB/s, a large copy's rate (two
// and four anchors per thread 34.5 and 37.4 us).
extern "C" __global__ __launch_bounds__(256) void vrs_detect_stage1(vrs_det1_args a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)a.B * a.A) return;
  const int b = (int)(i / a.A), ai = (int)(i - (int64_t)b * a.A);
  int s = 0;
  while (s + 1 < a.nscales && ai >= a.a_base[s + 1]) ++s;
  const int as = (s + 1 < a.nscales ? a.a_base[s + 1] : a.A) - a.a_base[s];
  const int j = ai - a.a_base[s];
  const float* sc = a.scores + (int64_t)b * a.nc * a.A + (int64_t)a.nc * a.a_base[s] + j;

  float xm = sc[0], sec = -INFINITY;   // largest and second largest logit
  int bc = 0;
  bool nan = xm != xm;
  auto see = [&](float x, int c) {
    sec = fmaxf(sec, fminf(x, xm));
    bc = x >= xm ? c : bc;
    xm = fmaxf(xm, x);
    nan |= x != x;
  };
  int c = 1;
  for (; c + 8 <= a.nc; c += 8) {
    float x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = sc[(int64_t)(c + u) * as];
#pragma unroll
    for (int u = 0; u < 8; ++u) see(x[u], c + u);
  }
  for (; c < a.nc; ++c) see(sc[(int64_t)c * as], c);

  const float near = fminf(xm - (xm < 0.0f ? 2e-5f : 1e-3f), 5.0f);
  const bool all = nan || xm < -80.0f;
  float best;
  if (all || sec >= near) {
    best = -1.0f;
    for (int c0 = 0; c0 < a.nc; c0 += 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = sc[(int64_t)min(c0 + u, a.nc - 1) * as];
      for (int u = 0; u < 8 && c0 + u < a.nc; ++u) {
        if (!all && x[u] < near) continue;
        const float p = 1.0f / (1.0f + expf(-x[u]));
        if (!(best > p)) { best = p; bc = c0 + u; }
      }
    }
  } else {
    best = 1.0f / (1.0f + expf(-xm));
  }
  const bool keep = best >= a.thr;
  a.keys[i] = keep ? (((uint64_t)__float_as_uint(best)) << 32) | (uint64_t)(0xffffffffu - (uint32_t)ai) : 0ull;
  if (!keep) return;   // nothing reads the other anchors' boxes and classes
  const float st = a.stride[s];
  const float* bb = a.boxes + (int64_t)b * 4 * a.A + 4 * (int64_t)a.a_base[s];
  const float l = bb[j], t = bb[as + j], r = bb[2 * as + j], bo = bb[3 * as + j];
  const float cx = ((float)(j % a.fw[s]) + 0.5f) * st;
  const float cy = ((float)(j / a.fw[s]) + 0.5f) * st;
  *reinterpret_cast<f32x4_any*>(a.xywh + i * 4) =
      (f32x4_any){cx + st * (r - l) * 0.5f, cy + st * (bo - t) * 0.5f, st * (l + r), st * (t + bo)};
  a.cls[i] = bc;
}

// One workgroup per image, 64 of them at bs64: the time is its chain of
// dependent steps.  The keys stay in registers (16 per thread; images of more
// than 16384 anchors read the rest again per digit); a digit is 11 bits (16
// bins per octave of the score: 8-bit digits put most keys into two bins, whose
// LDS atomics then queue up) and its bin is found by a parallel scan (one
// thread walking 256 bins took 10 us); the sort keeps one key per thread and
// crosses lanes inside a wave.  39.5 -> 15.5 us at 8400 anchors, nearly
// all kept (threshold 0.001).
namespace {
constexpr int TOPK_MAX = 1024;
constexpr int KEY_REGS = 16;
constexpr int DIGIT = 11, BINS = 1 << DIGIT;
}

extern "C" __global__ __launch_bounds__(1024) void vrs_detect_stage2(vrs_det2_args a) {
  __shared__ uint32_t hist[BINS];
  __shared__ uint64_t sel[TOPK_MAX];
  __shared__ uint32_t s_wave[16], s_nsel, s_digit, s_krem, s_ntop;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t* keys = a.keys + (int64_t)b * a.A;

  uint64_t reg[KEY_REGS];
#pragma unroll
  for (int r = 0; r < KEY_REGS; ++r) reg[r] = tid + r * 1024 < a.A ? keys[tid + r * 1024] : 0ull;
  auto each_key = [&](auto f) {   // whole waves together (f may use ballots)
#pragma unroll
    for (int r = 0; r < KEY_REGS; ++r)
      if (r * 1024 < a.A) f(reg[r]);
    for (int i0 = KEY_REGS * 1024; i0 < a.A; i0 += 1024) f(i0 + tid < a.A ? keys[i0 + tid] : 0ull);
  };
  // inclusive sum over the workgroup's threads; two barriers
  auto block_scan = [&](uint32_t v) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t u = __shfl_up(v, d);
      if (lane >= d) v += u;
    }
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) before += w < wave ? s_wave[w] : 0u;
    __syncthreads();
    return v + before;
  };

  uint32_t local = 0;
  each_key([&](uint64_t key) { local += key != 0ull; });
  const uint32_t upto = block_scan(local);
  if (tid == 1023) s_krem = upto;
  if (tid == 0) s_nsel = 0;
  __syncthreads();
  const uint32_t count = s_krem;
  const uint32_t k = count < (uint32_t)a.max_det ? count : (uint32_t)a.max_det;

  // gather threshold: every nonzero key when they all fit the buffer
  uint64_t thr_key = 1ull;
  if (count > (uint32_t)TOPK_MAX && k > 0) {
    uint64_t prefix = 0, pmask = 0;
    uint32_t krem = k;
    // scores are at most 1.0f: bits 62 and 63 of a key are zero
    for (int shift = 62 - DIGIT; ; shift = shift > DIGIT ? shift - DIGIT : 0) {
      hist[tid] = 0;
      hist[tid + 1024] = 0;
      __syncthreads();
      each_key([&](uint64_t key) {
        if (key != 0ull && (key & pmask) == prefix) atomicAdd(&hist[(uint32_t)(key >> shift) & (BINS - 1)], 1u);
      });
      __syncthreads();
      // thread t scans bins BINS-1-2t and BINS-2-2t, from the top down
      const uint32_t hi = hist[BINS - 1 - 2 * tid], lo = hist[BINS - 2 - 2 * tid];
      const uint32_t incl = block_scan(hi + lo), excl = incl - hi - lo;
      if (excl < krem && krem <= incl) {   // one thread: the bin of the krem-th key
        const bool top = krem <= excl + hi;
        const uint32_t above = top ? excl : excl + hi;
        s_digit = (uint32_t)(BINS - 1 - 2 * tid) - (top ? 0u : 1u);
        s_krem = krem - above;
        // keys whose digits so far are >= the new prefix: above it at the
        // earlier digits (k - krem), in the higher bins of this one and in it
        s_ntop = (k - krem) + above + (top ? hi : lo);
      }
      __syncthreads();
      krem = s_krem;
      prefix |= ((uint64_t)s_digit) << shift;
      pmask |= ((uint64_t)(BINS - 1)) << shift;
      const bool fits = s_ntop <= (uint32_t)TOPK_MAX;
      __syncthreads();
      if (fits || shift == 0) break;
    }
    // lower bits zero: the keys >= prefix are exactly those counted in s_ntop,
    // and they include the k largest
    thr_key = prefix;
  }

  sel[tid] = 0ull;
  __syncthreads();
  if (k > 0)
    each_key([&](uint64_t key) {
      const bool in = key != 0ull && key >= thr_key;
      const uint64_t m = __ballot(in);
      uint32_t base = 0;
      if (lane == 0 && m) base = atomicAdd(&s_nsel, (uint32_t)__popcll(m));
      base = __shfl(base, 0);
      const uint32_t slot = base + (uint32_t)__popcll(m & ((1ull << lane) - 1));
      if (in && slot < (uint32_t)TOPK_MAX) sel[slot] = key;
    });
  __syncthreads();
  // sort the smallest power of two of slots holding every gathered key
  const uint32_t nsel = s_nsel < (uint32_t)TOPK_MAX ? s_nsel : (uint32_t)TOPK_MAX;
  int P = 2;
  while ((uint32_t)P < nsel) P <<= 1;

  // bitonic sort, descending, over P slots (zeros sink to the end): thread t
  // holds slot t; partners in the same wave by shuffle, others through LDS
  uint64_t el = sel[tid];
  for (int size = 2; size <= P; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      uint64_t y;
      if (stride >= 64) {
        __syncthreads();
        sel[tid] = el;
        __syncthreads();
        y = sel[tid ^ stride];
      } else {
        y = __shfl_xor((unsigned long long)el, stride);
      }
      const bool larger = ((tid & stride) == 0) == ((tid & size) == 0);
      el = (el > y) == larger ? el : y;
    }

  if (tid == 0) a.count[b] = (int32_t)k;
  if (tid < a.max_det) {   // max_det <= 1024 (host)
    const int64_t o = (int64_t)b * a.max_det + tid;
    if ((uint32_t)tid < k) {
      const int anchor = (int)(0xffffffffu - (uint32_t)(el & 0xffffffffull));
      a.out_score[o] = __uint_as_float((uint32_t)(el >> 32));
      a.out_anchor[o] = anchor;
      a.out_cls[o] = a.cls[(int64_t)b * a.A + anchor];
      const f32x4_any xy = *reinterpret_cast<const f32x4_any*>(a.xywh + ((int64_t)b * a.A + anchor) * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) a.out_xywh[o * 4 + q] = xy[q];
    } else {
      a.out_score[o] = 0.f;
      a.out_anchor[o] = -1;
      a.out_cls[o] = -1;
#pragma unroll
      for (int q = 0; q < 4; ++q) a.out_xywh[o * 4 + q] = 0.f;
    }
  }
}

// Letterbox pixels -> [cx, cy, w, h] normalised to the original image, the
// reference's un-letterbox (examples/yolo26.rs:1531-1547) in the same float32
// operations: s = img / max(ow, oh); new = round(o * s) (half away from
// zero); pad = (img - new) / 2 in integers; divide by o * s.  One thread per
// detection slot; slots past count[b] are zeroed.
extern "C" __global__ __launch_bounds__(256) void vrs_detect_unletterbox(vrs_unlb_args a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)a.B * a.max_det) return;
  const int b = (int)(i / a.max_det), k = (int)(i - (int64_t)b * a.max_det);
  float* o = a.out + i * 4;
  if (k >= a.count[b]) {
    o[0] = o[1] = o[2] = o[3] = 0.f;
    return;
  }
  const int ow = a.orig_wh[2 * b], oh = a.orig_wh[2 * b + 1];
  const float s = (float)a.img_size / (float)(ow > oh ? ow : oh);
  const int nw = (int)roundf((float)ow * s), nh = (int)roundf((float)oh * s);
  const float px = (float)(a.img_size > nw ? (a.img_size - nw) / 2 : 0);
  const float py = (float)(a.img_size > nh ? (a.img_size - nh) / 2 : 0);
  const float sx = (float)ow * s, sy = (float)oh * s;
  const float* d = a.xywh + i * 4;
  o[0] = (d[0] - px) / sx;
  o[1] = (d[1] - py) / sy;
  o[2] = d[2] / sx;
  o[3] = d[3] / sy;
}

// ---- letterbox preprocessing (examples/yolo26.rs:1229-1253) ---------------
// preprocess_image_raw resizes with image 0.25.10 imageops::resize(...,
// FilterType::Triangle): a vertical pass over the source columns into float32
// (weights normalised per output row), then a horizontal pass over that
// buffer (normalised per output column), clamped to [0, 255] and rounded half
// away from zero to u8; the canvas holds u8 / 255 inside the resized region
// and 114 / 255 elsewhere.  Per axis, output index o of a dst-long axis from a
// src-long one: ratio = src / dst, sr = max(ratio, 1), centre = (o + 0.5) *
// ratio, taps i in [clamp(floor(centre - sr), 0, src - 1), clamp(ceil(centre
// + sr), lo + 1, src)), weight tri((i - (centre - 0.5)) / sr) / sum, tri(x) =
// max(0, 1 - |x|).  The kernel fuses both passes per output pixel with the
// same float32 operations in the same order (vertical sum over a column's
// taps, then the horizontal sum over columns), so it reproduces the two-pass
// result bit for bit; contraction into FMA is off as in the reference.
namespace {
__device__ inline float lb_tri(float x) {
  const float a = fabsf(x);
  return a < 1.0f ? 1.0f - a : 0.0f;
}
// Window [lo, hi) of output index o along an axis of src source pixels, ratio
// of them to an output pixel; at most `cap` taps (the host's ratio bounds keep
// the true window within it).  c, sr: the weights' centre and support.
__device__ inline void lb_bounds(int o, int src, float ratio, int cap, int& lo, int& hi, float& c, float& sr) {
#pragma clang fp contract(off)
  sr = ratio < 1.0f ? 1.0f : ratio;  // support 1 x sratio
  const float centre = ((float)o + 0.5f) * ratio;
  lo = (int)floorf(centre - sr);
  lo = lo < 0 ? 0 : (lo > src - 1 ? src - 1 : lo);
  hi = (int)ceilf(centre + sr);
  hi = hi < lo + 1 ? lo + 1 : (hi > src ? src : hi);
  if (hi - lo > cap) hi = lo + cap;
  c = centre - 0.5f;
}
// The window of output index o with its normalised weights written to
// w[0..n) and zeros to w[n..fill); returns n.  One division per tap for the weight and one for the
// normalisation, as the reference does them.
__device__ inline int lb_window(int o, int src, int dst, int cap, float* w, int& lo, int fill = 0) {
#pragma clang fp contract(off)
  int h;
  float c, sr;
  lb_bounds(o, src, (float)src / (float)dst, cap, lo, h, c, sr);
  float sum = 0.0f;
  for (int i = lo; i < h; ++i) {
    const float v = lb_tri(((float)i - c) / sr);
    w[i - lo] = v;
    sum += v;
  }
  for (int i = 0; i < h - lo; ++i) w[i] = w[i] / sum;
  for (int i = h - lo; i < fill; ++i) w[i] = 0.0f;
  return h - lo;
}
// Clamp, round half away from zero, / 255.  The quotient of a whole number in
// 0..255 by 255, correctly rounded: a product with the rounded reciprocal and
// one residual step (Markstein), equal to the division for all 256.
__device__ inline float lb_quant(float v) {
  v = v < 0.0f ? 0.0f : (v > 255.0f ? 255.0f : v);
  float q = truncf(v);
  if (v - q >= 0.5f) q += 1.0f;
  const float rcp = 1.0f / 255.0f, y = q * rcp;
  return __builtin_fmaf(__builtin_fmaf(-255.0f, y, q), rcp, y);
}
constexpr int LB_TW = 64, LB_TH = 4, LB_LD = VRS_LB_MAX_TAPS + 1;  // odd row pitch: no bank conflicts
}  // namespace

// One workgroup per 64 x 4 tile of one image's canvas (grid.y = image).  The
// 64 column and 4 row windows of the tile are computed once into LDS; each
// thread then sums its pixel's window from the RGB8 source (all three
// channels per tap) and writes the three NCHW planes.
extern "C" __global__ __launch_bounds__(256) void vrs_letterbox_f32(vrs_lb_args a) {
#pragma clang fp contract(off)
  __shared__ float wcol[LB_TW * LB_LD];
  __shared__ float wrow[LB_TH * LB_LD];
  __shared__ int gcol[LB_TW][2], grow[LB_TH][2];
  const vrs_lb_image im = a.img[blockIdx.y];
  const int tiles_x = (a.S + LB_TW - 1) / LB_TW;
  const int x0 = (int)(blockIdx.x % tiles_x) * LB_TW, y0 = (int)(blockIdx.x / tiles_x) * LB_TH;
  const int tx = threadIdx.x % LB_TW, ty = threadIdx.x / LB_TW;
  // does the tile meet the resized region? (uniform over the workgroup)
  const bool inside = x0 < im.px + im.nw && x0 + LB_TW > im.px && y0 < im.py + im.nh && y0 + LB_TH > im.py;
  if (inside) {
    const int t = threadIdx.x;
    if (t < LB_TW) {
      const int p = x0 + t - im.px;
      if (p >= 0 && p < im.nw) {
        int lo;
        const int n = lb_window(p, im.w, im.nw, VRS_LB_MAX_TAPS, wcol + t * LB_LD, lo);
        gcol[t][0] = lo;
        gcol[t][1] = lo + n;
      }
    } else if (t < LB_TW + LB_TH) {
      const int r = t - LB_TW, p = y0 + r - im.py;
      if (p >= 0 && p < im.nh) {
        int lo;
        const int n = lb_window(p, im.h, im.nh, VRS_LB_MAX_TAPS, wrow + r * LB_LD, lo);
        grow[r][0] = lo;
        grow[r][1] = lo + n;
      }
    }
    __syncthreads();
  }
  const int ox = x0 + tx, oy = y0 + ty;
  if (ox >= a.S || oy >= a.S) return;
  const int64_t plane = (int64_t)a.S * a.S;
  float* o = a.out + (int64_t)im.slot * 3 * plane + (int64_t)oy * a.S + ox;
  const int px = ox - im.px, py = oy - im.py;
  if (!inside || px < 0 || px >= im.nw || py < 0 || py >= im.nh) {
    o[0] = a.pad;
    o[plane] = a.pad;
    o[2 * plane] = a.pad;
    return;
  }
  const int lo = gcol[tx][0], hi = gcol[tx][1], top = grow[ty][0], bot = grow[ty][1];
  const int64_t row = (int64_t)im.w * 3;
  const uint8_t* src = a.rgb + im.off + (int64_t)top * row;
  const float* wy = wrow + ty * LB_LD;
  const float* wx = wcol + tx * LB_LD;
  float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
  const int n = bot - top;
  for (int i = lo; i < hi; ++i) {
    const uint8_t* p = src + (int64_t)i * 3;
    float t0 = 0.0f, t1 = 0.0f, t2 = 0.0f;
    for (int j0 = 0; j0 < n; j0 += 8) {   // 8 taps' bytes in flight, then the sums in order
      uint8_t q[8][3];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j0 + j < n) {
          const uint8_t* pj = p + (int64_t)(j0 + j) * row;
          q[j][0] = pj[0];
          q[j][1] = pj[1];
          q[j][2] = pj[2];
        }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j0 + j < n) {
          const float w = wy[j0 + j];
          t0 += (float)q[j][0] * w;
          t1 += (float)q[j][1] * w;
          t2 += (float)q[j][2] * w;
        }
    }
    const float w = wx[i - lo];
    s0 += t0 * w;
    s1 += t1 * w;
    s2 += t2 * w;
  }
  o[0] = lb_quant(s0);
  o[plane] = lb_quant(s1);
  o[2 * plane] = lb_quant(s2);
}

// Staged variants for images enlarged or kept (vrs_letterbox_f32_s1), or shrunk
// at most 2x (_s2), 4x (_s4) or VRS_LB_STAGED_RATIO = 8x (_s8) per axis: one
// workgroup per TW x TH tile.  The source patch the tile reads (rows spanned by its row windows x
// columns spanned by its column windows) is copied into LDS with aligned
// 16-byte loads, all in flight together, while the windows' weights are
// computed; the vertical pass then runs once per (tile row, source column)
// from LDS into a float32 buffer, and the horizontal pass reads that buffer --
// the same float32 operations in the same order as the direct kernel and the
// two-pass reference.
//
// LDS instructions bound the vertical pass when it reads single bytes, so a
// thread takes four pixels of a row: 12 bytes, as dwords shifted into place by
// the row's misalignment.  Windows are padded with weights of zero to a fixed
// length, so that a window's reads are all in flight (a sum of products >= 0
// is unchanged by adding +0); what the padding reads is some byte of the patch
// or a sum of them, so finite.  A window holds at most 2 R + 1 taps: its real
// interval is 2 R long, and rounding a bound never moves it past a whole number.
// Measured (single bytes and 4 rows a tile -> dwords and 8 rows at R <= 2): 16
// frames of 1280 x 720 to 640 52.2 -> 40.6 us (4 rows 50.9, 16 rows 40.6, 128
// columns 39.7), 1920 x 1080 108 -> 95, 4 of 3200 x 2160 to 640 166 -> 118.
// VALU and LDS issue bound the small ratios (about 130 vector instructions an
// output pixel at five taps), hence the instance of three taps (R = 1): 32
// frames of 640 x 480 to 640 105 -> 63 us (78 on the 2x instance), 8 of 400 x
// 300 to 1280 95.5 -> 48.6 (60.5; 3.3 TB/s).
namespace {
// R: the largest shrink factor per axis the instance accepts; LDS is sized
// for it, so the small-ratio instance fits more workgroups per CU
template <int R, int TW, int TH, int NT>
__device__ __forceinline__ void lb_staged(const vrs_lb_args& a) {
#pragma clang fp contract(off)
  constexpr int TAPS = 2 * R + 1, U = R == 2 ? 5 : R <= 4 ? 3 : 6;   // taps in flight
  constexpr int PAD = (TAPS + U - 1) / U * U;                          // padded window
  // weights: a window per thread, or, of more taps, a tap (17 taps: 34 divisions
  // in a row, 338 us for 16 frames of 3100 x 2400 to 416; by tap 295, but 41.5
  // instead of 40.9 at 5 taps)
  constexpr bool BY_TAP = R > 4;
  constexpr int LDC = PAD | 1, LDR = (PAD + 3) / 4 * 4;
  // source columns / rows a tile touches: (n - 1) * ratio + 2 * ratio + 2, +2 slack
  constexpr int CMAX = (TW - 1) * R + 2 * R + 4;
  constexpr int RMAX = (TH - 1) * R + 2 * R + 4;
  constexpr int VU = (CMAX + U + 3) / 4;               // units of 4 pixels, the padding's reads included
  constexpr int PW = (15 + 12 * VU + 4 + 15) / 16;     // 16-byte chunks per patch row (15-byte lead-in)
  constexpr int CL = PW <= 32 ? 32 : 64;               // lanes that copy one row
  constexpr int RPR = NT / CL, ROUNDS = (RMAX + RPR - 1) / RPR, VREG = ROUNDS < 4 ? ROUNDS : 4;
  static_assert(PW <= 64 && TW + TH <= NT && NT % TW == 0, "tile");
  __shared__ float wcol[TW * LDC];
  __shared__ __attribute__((aligned(16))) float wrow[TH * LDR];
  __shared__ int gcol[TW][2], grow[TH][2];
  __shared__ u32x4_t patch[RMAX * PW];
  __shared__ __attribute__((aligned(16))) float vbuf[TH * VU * 12];
  float* const raw = vbuf;                             // the unnormalised weights, before the vertical pass
  static_assert((TW + TH) * PAD <= TH * VU * 12, "weights fit");
  const vrs_lb_image im = a.img[blockIdx.y];
  const int tiles_x = (a.S + TW - 1) / TW;
  const int x0 = (int)(blockIdx.x % tiles_x) * TW, y0 = (int)(blockIdx.x / tiles_x) * TH;
  const int64_t plane = (int64_t)a.S * a.S;
  float* ob = a.out + (int64_t)im.slot * 3 * plane;
  const int t = threadIdx.x;
  const int tx = t % TW, ty = t / TW;
  const int ox = x0 + tx;
  // in-image columns [cf, cl] and rows [rf, rl] of the tile (uniform)
  const int cf = max(im.px - x0, 0), cl = min(im.px + im.nw - x0, TW) - 1;
  const int rf = max(im.py - y0, 0), rl = min(im.py + im.nh - y0, TH) - 1;
  if (cf > cl || rf > rl) {   // all padding
    for (int r = ty; r < TH; r += NT / TW) {
      if (ox >= a.S || y0 + r >= a.S) continue;
      float* o = ob + (int64_t)(y0 + r) * a.S + ox;
      o[0] = a.pad;
      o[plane] = a.pad;
      o[2 * plane] = a.pad;
    }
    return;
  }
  // window bounds are non-decreasing along an axis: the patch is source rows
  // [top of the first row window, bottom of the last) x columns [lo of the
  // first column window, hi of the last)
  int c_lo, ytop, hi, skip;
  float f0, f1;
  const float ratio_x = (float)im.w / (float)im.nw, ratio_y = (float)im.h / (float)im.nh;
  lb_bounds(x0 + cf - im.px, im.w, ratio_x, TAPS, c_lo, skip, f0, f1);
  lb_bounds(x0 + cl - im.px, im.w, ratio_x, TAPS, skip, hi, f0, f1);
  const int ncol = min(hi - c_lo, CMAX);   // <= CMAX and RMAX by the ratio bound
  lb_bounds(y0 + rf - im.py, im.h, ratio_y, TAPS, ytop, skip, f0, f1);
  lb_bounds(y0 + rl - im.py, im.h, ratio_y, TAPS, skip, hi, f0, f1);
  const int nrow = min(hi - ytop, RMAX);
  // patch row i holds the source bytes [s_i, s_i + 3*ncol) of image row
  // ytop + i (s_i = off + ((ytop + i)*w + c_lo)*3), copied as the 16-byte
  // aligned chunks that cover them, so its bytes start at s_i's address mod
  // 16.  Chunks straddling the image's first or last byte (only those) are
  // assembled from byte loads.
  const unsigned char* img0 = a.rgb + im.off;
  const unsigned char* img1 = img0 + (int64_t)im.w * im.h * 3;
  const unsigned char* src = img0 + ((int64_t)ytop * im.w + c_lo) * 3;
  const int64_t stride = (int64_t)im.w * 3;
  const uint32_t lead0 = (uint32_t)(reinterpret_cast<uintptr_t>(src) & 15), dlead = (uint32_t)stride;
  const int nq = (3 * ncol + 15 + 15) / 16;   // chunks per row copy (<= PW)
  const int cd = t % CL, cr = t / CL;
#pragma unroll 1
  for (int base = 0; base < ROUNDS; base += VREG) {
    u32x4_t v[VREG];
#pragma unroll
    for (int u = 0; u < VREG; ++u) {
      const int i = cr + (base + u) * RPR;
      v[u] = (u32x4_t){0, 0, 0, 0};
      if (i < nrow && cd < nq) {
        const unsigned char* q = reinterpret_cast<const unsigned char*>(
            (reinterpret_cast<uintptr_t>(src + i * stride) & ~(uintptr_t)15) + 16 * (uintptr_t)cd);
        if (q >= img0 && q + 16 <= img1) {
          v[u] = *reinterpret_cast<const u32x4_t*>(q);
        } else {
          uint32_t wv[4] = {0, 0, 0, 0};
          for (int k = 0; k < 16; ++k)
            if (q + k >= img0 && q + k < img1) wv[k / 4] |= (uint32_t)q[k] << (8 * (k % 4));
          v[u] = (u32x4_t){wv[0], wv[1], wv[2], wv[3]};
        }
      }
    }
    if (base == 0) {   // the windows, under the first loads
      if constexpr (BY_TAP) {   // a tap per thread, zero past a window's end
        for (int k = t; k < (TW + TH) * PAD; k += NT) {
          const int g = k / PAD, i = k - g * PAD;
          const bool col = g < TW;
          const int p = col ? x0 + g - im.px : y0 + g - TW - im.py;
          float v = 0.0f;
          if (p >= 0 && p < (col ? im.nw : im.nh)) {
            int lo, h;
            float c, sr;
            lb_bounds(p, col ? im.w : im.h, col ? ratio_x : ratio_y, TAPS, lo, h, c, sr);
            if (i < h - lo) v = lb_tri(((float)(lo + i) - c) / sr);
            if (i == 0) {
              int* e = col ? gcol[g] : grow[g - TW];
              e[0] = lo - (col ? c_lo : ytop);
              e[1] = h - lo;
            }
          }
          raw[k] = v;
        }
        __syncthreads();
        for (int k = t; k < (TW + TH) * PAD; k += NT) {
          const int g = k / PAD, i = k - g * PAD;
          float sum = 0.0f;
#pragma unroll
          for (int e = 0; e < PAD; ++e) sum += raw[g * PAD + e];
          (g < TW ? wcol + g * LDC : wrow + (g - TW) * LDR)[i] = raw[k] / sum;
        }
      } else if (t < TW) {
        if (t >= cf && t <= cl) {
          int lo;
          gcol[t][1] = lb_window(x0 + t - im.px, im.w, im.nw, TAPS, wcol + t * LDC, lo, PAD);
          gcol[t][0] = lo - c_lo;
        }
      } else if (t < TW + TH) {
        const int r = t - TW;
        if (r >= rf && r <= rl) {
          int lo;
          grow[r][1] = lb_window(y0 + r - im.py, im.h, im.nh, TAPS, wrow + r * LDR, lo, PAD);
          grow[r][0] = lo - ytop;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < VREG; ++u) {
      const int i = cr + (base + u) * RPR;
      if (i < nrow && cd < nq) patch[i * PW + cd] = v[u];
    }
  }
  __syncthreads();
  // vertical pass: one unit of four source columns of a tile row per thread
  // and step, the columns that the horizontal padding reads included
  const uint32_t* pd = reinterpret_cast<const uint32_t*>(patch);
  const int nu = min((ncol + U + 3) / 4, VU);
  const int units = (rl - rf + 1) * nu;
  const float inv_nu = 1.0f / (float)nu;
  for (int idx = t; idx < units; idx += NT) {
    int u;
    const int r = rf + fdivmod(idx, nu, inv_nu, u);
    const int top = grow[r][0], n = grow[r][1];
    const float* wy = wrow + r * LDR;
    float acc[12];
#pragma unroll
    for (int e = 0; e < 12; ++e) acc[e] = 0.0f;
#pragma unroll
    for (int j0 = 0; j0 < PAD; j0 += U) {
      if (j0 >= n) break;
      uint32_t q[U][4], sh[U];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int i = min(top + j0 + j, nrow - 1);
        const uint32_t lead = (lead0 + (uint32_t)i * dlead) & 15;
        const uint32_t* p = pd + i * (PW * 4) + (lead >> 2) + 3 * u;
        sh[j] = lead & 3;
#pragma unroll
        for (int e = 0; e < 4; ++e) q[j][e] = p[e];
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const float w = wy[j0 + j];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          const uint32_t d = __builtin_amdgcn_alignbyte(q[j][e + 1], q[j][e], sh[j]);
          acc[4 * e + 0] += (float)(d & 0xff) * w;
          acc[4 * e + 1] += (float)(d >> 8 & 0xff) * w;
          acc[4 * e + 2] += (float)(d >> 16 & 0xff) * w;
          acc[4 * e + 3] += (float)(d >> 24) * w;
        }
      }
    }
    f32x4_t* vv = reinterpret_cast<f32x4_t*>(vbuf + (r * VU + u) * 12);
#pragma unroll
    for (int e = 0; e < 3; ++e) vv[e] = (f32x4_t){acc[4 * e], acc[4 * e + 1], acc[4 * e + 2], acc[4 * e + 3]};
  }
  __syncthreads();
  // horizontal pass: a column per thread, its weights held over the rows
  if (ox >= a.S) return;
  const bool in_x = tx >= cf && tx <= cl;
  const int lo = in_x ? gcol[tx][0] : 0, n = in_x ? min(gcol[tx][1], ncol - lo) : 0;
#pragma unroll
  for (int r0 = 0; r0 < TH; r0 += NT / TW) {
    const int r = r0 + ty;
    if (y0 + r >= a.S) continue;
    float* o = ob + (int64_t)(y0 + r) * a.S + ox;
    if (!in_x || r < rf || r > rl) {
      o[0] = a.pad;
      o[plane] = a.pad;
      o[2 * plane] = a.pad;
      continue;
    }
    const float* vv = vbuf + r * (VU * 12) + lo * 3;
    const float* wx = wcol + tx * LDC;
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int i0 = 0; i0 < PAD; i0 += U) {
      if (i0 >= n) break;
#pragma unroll
      for (int i = i0; i < i0 + U; ++i) {
        const float w = wx[i];
        s0 += vv[3 * i] * w;
        s1 += vv[3 * i + 1] * w;
        s2 += vv[3 * i + 2] * w;
      }
    }
    o[0] = lb_quant(s0);
    o[plane] = lb_quant(s1);
    o[2 * plane] = lb_quant(s2);
  }
}
}  // namespace

extern "C" __global__ __launch_bounds__(256) void vrs_letterbox_f32_s1(vrs_lb_args a) { lb_staged<1, 64, 8, 256>(a); }
extern "C" __global__ __launch_bounds__(256) void vrs_letterbox_f32_s2(vrs_lb_args a) { lb_staged<2, 64, 8, 256>(a); }
extern "C" __global__ __launch_bounds__(256) void vrs_letterbox_f32_s4(vrs_lb_args a) { lb_staged<4, 64, 4, 256>(a); }
// 32 x 4 tiles (128 threads) keep the patch of an 8x shrink within 40 KB of LDS
extern "C" __global__ __launch_bounds__(128) void vrs_letterbox_f32_s8(vrs_lb_args a) {
  lb_staged<VRS_LB_STAGED_RATIO, 32, 4, 128>(a);
}

// Grid-unit decode on [B,4,A] rows l,t,r,b (kernels/detect_decode.rs:36-86):
// cx = (ax - l + ax + r) * 0.5 * s, cy likewise, w = (r + l) * s, h = (b + t) * s.
extern "C" __global__ __launch_bounds__(256) void vrs_detect_decode_grid(vrs_dec_args a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)a.B * a.A) return;
  const int b = (int)(i / a.A), ai = (int)(i - (int64_t)b * a.A);
  const float* bx = a.boxes + (int64_t)b * 4 * a.A;
  float* o = a.out + (int64_t)b * 4 * a.A;
  const float x1 = a.ax[ai] - bx[ai], y1 = a.ay[ai] - bx[a.A + ai];
  const float x2 = a.ax[ai] + bx[2 * a.A + ai], y2 = a.ay[ai] + bx[3 * a.A + ai];
  const float s = a.st[ai];
  o[ai] = (x1 + x2) * 0.5f * s;
  o[a.A + ai] = (y1 + y2) * 0.5f * s;
  o[2 * a.A + ai] = (x2 - x1) * s;
  o[3 * a.A + ai] = (y2 - y1) * s;
}
