"""Parity of kernels and dispatch rules at the sizes where they change hands:
tile edges, remainders, unaligned views, the smallest and largest of a range."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import ctx, rounder, tdtype, vrs

pytestmark = pytest.mark.gpu
DT = [pytest.param(vrs.F32, id="f32"), pytest.param(vrs.BF16, id="bf16")]


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("n,c,c_pad,h,w,shift", [
    (2, 3, 8, 16, 32, 0),      # the 8-channel tile, one whole tile
    (1, 3, 8, 19, 27, 0),      # its last partial tile, single-pixel accesses (513 pixels)
    (1, 3, 3, 5, 7, 0),        # rows that no 16-byte chunk fits
    (2, 64, 64, 8, 8, 0),      # the 64-channel tile, one whole tile
    (1, 65, 72, 5, 13, 0),     # 65 pixels and channels: both remainders, padded rows
    (1, 130, 130, 4, 4, 1),    # unaligned rows and an image base off 16 bytes
])
def test_layout_conversions_exact(dtype, n, c, c_pad, h, w, shift):
    """NCHW float32 -> NHWC and back are copies (one rounding to the element type)."""
    import torch
    rng = np.random.default_rng(21)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    x[0, 0, 0, 0], x[0, -1, -1, -1] = np.inf, -0.0
    flat = torch.zeros(shift + x.size, device="cuda")
    xt = flat[shift:].view(n, c, h, w)
    xt.copy_(torch.from_numpy(x))
    y = torch.full((n, h, w, c_pad), 7.0, dtype=tdtype(dtype), device="cuda")
    ctx().pack_input(xt, vrs.nhwc(y), dtype)
    torch.cuda.synchronize()
    want = np.zeros((n, h, w, c_pad), np.float32)
    want[..., :c] = rounder(dtype)(x).transpose(0, 2, 3, 1)
    assert np.array_equal(y.float().cpu().numpy(), want)
    # back from a channel slice (offset 1 when there is room: unaligned) and from the whole buffer
    for off in (0, 1):
        back = torch.full((shift + n * (c - off) * h * w,), 9.0, device="cuda")
        ctx().unpack_output(vrs.nhwc(y, c - off, off), dtype, back[shift:].view(n, c - off, h, w))
        torch.cuda.synchronize()
        assert np.array_equal(back[shift:].cpu().numpy().reshape(n, c - off, h, w), rounder(dtype)(x)[:, off:])


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("n,c,c_pad,h,w,shift", [
    (1027, 3, 8, 1, 1, 0), (1100, 7, 8, 8, 7, 0),     # 8-channel tiles
    (1103, 5, 5, 5, 1, 1), (262145, 5, 5, 1, 1, 1),   # rows that no 16-byte chunk fits, an unaligned base; 512 to a tile
    (700, 130, 136, 1, 1, 0), (603, 64, 68, 3, 5, 0),  # 64-channel tiles, a last one of padding alone
    (2050, 130, 136, 7, 1, 0), (1050, 9, 9, 3, 7, 1),
])
def test_layout_conversions_of_small_maps(dtype, n, c, c_pad, h, w, shift):
    """Small maps, whole images to a tile: copies, as the larger ones."""
    test_layout_conversions_exact(dtype, n, c, c_pad, h, w, shift)


@pytest.mark.parametrize("n,c,h,w", [(1 << 24, 3, 1, 1), ((1 << 24) + 3, 9, 11, 3)])
def test_layout_conversions_of_many_maps(n, c, h, w):
    """2^24 maps and more: calls that take several launches (64-channel tiles of one image)."""
    import torch
    part = torch.randn(1 << 12, c, h, w, device="cuda")
    x = torch.empty(n, c, h, w, device="cuda")
    for i in range(0, n, 1 << 12):
        x[i:i + (1 << 12)] = part[:min(1 << 12, n - i)]
    c_pad = (c + 7) // 8 * 8
    y = torch.empty(n, h, w, c_pad, dtype=torch.bfloat16, device="cuda")
    ctx().pack_input(x, vrs.nhwc(y), vrs.BF16)
    x.zero_()
    ctx().unpack_output(vrs.nhwc(y, c), vrs.BF16, x)
    want = part.bfloat16().float()
    for i in range(0, n, 1 << 12):
        assert torch.equal(x[i:i + (1 << 12)], want[:min(1 << 12, n - i)])


SPLIT_TILES = [pytest.param(vrs.TILE_KW16 | vrs.TILE_SPLIT_1, id="16x4"),
               pytest.param(vrs.TILE_KW16 | vrs.TILE_SPLIT_4, id="16w4"),
               pytest.param(vrs.TILE_KW16 | vrs.TILE_SPLIT_8, id="16w8"),
               pytest.param(vrs.TILE_KW32 | vrs.TILE_SPLIT_4, id="32w4"),
               pytest.param(vrs.TILE_KW32 | vrs.TILE_SPLIT_8, id="32w8")]


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("tile", SPLIT_TILES)
@pytest.mark.parametrize("case", [
    # n, cin, h, w, cout, k, s, residual
    (1, 8, 1, 1, 4, 1, 1, False),       # one pixel, one chunk of K: most waves have no step
    (1, 8, 5, 3, 20, 3, 1, True),       # 15 pixels, 20 channels; taps of one chunk
    (2, 24, 4, 4, 36, 3, 2, False),     # taps that do not fill a step, 8 pixels
    (1, 32, 8, 8, 32, 3, 1, True),      # whole 32x32 tiles; float32: one step per tap
    (1, 64, 3, 11, 33 * 4, 3, 1, False),  # 33 pixels, bfloat16: one step per tap
    (3, 72, 6, 7, 64, 1, 1, True),      # 126 pixels: the last of four neighbouring tiles is partial
    (1, 128, 7, 9, 48, 5, 1, False),    # 25 taps
    (1, 512, 4, 5, 16, 3, 2, False),    # deep K: several rounds of steps per wave
])
def test_split_k_conv(case, tile, dtype):
    import zlib

    import oracle
    import torch
    from gpu_util import dev, from_nhwc, rel_err, to_nhwc
    n, cin, h, w, cout, k, s, with_res = case
    rnd = rounder(dtype)
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()))
    x = rnd(rng.standard_normal((n, cin, h, w)).astype(np.float32))
    wt = rnd((rng.standard_normal((cout, cin, k, k)) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32))
    scale = rng.uniform(0.5, 1.5, cout).astype(np.float32)
    shift = rng.normal(0, 0.2, cout).astype(np.float32)
    ho, wo = (h - 1) // s + 1, (w - 1) // s + 1
    ref = oracle.affine_act(oracle.conv2d(x, wt, s, k // 2), scale, shift, 1)
    res = rnd(rng.standard_normal(ref.shape).astype(np.float32)) if with_res else None
    xt = to_nhwc(x, dtype, cin + 8, 8)
    yt = torch.full((n, ho, wo, cout + 8), 7.0, dtype=tdtype(dtype), device="cuda")
    rt = to_nhwc(res, dtype, cout + 4, 4) if with_res else None
    ctx().conv2d(vrs.nhwc(xt, cin, 8), dev(vrs.pack_conv_weight(wt, 1, cin, dtype)), dev(scale), dev(shift),
                 vrs.nhwc(yt, cout, 4), k, s, 1, vrs.ACT_SILU, vrs.nhwc(rt, cout, 4) if with_res else None, dtype,
                 tile=tile)
    torch.cuda.synchronize()
    # the bounds of the other conv kernels (float32: eps * sqrt(K) products in another order)
    err = rel_err(from_nhwc(yt, cout, 4), ref + res if with_res else ref, 5e-2 if dtype == vrs.F32 else 1e-1)
    assert err < (1e-4 if dtype == vrs.F32 else 2e-2), err
    assert torch.all(yt[..., :4] == 7.0) and torch.all(yt[..., cout + 4:] == 7.0)


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("tile", SPLIT_TILES)
def test_split_k_network(tile, dtype):
    """Every dense conv of YOLO26n on a split-K tile (fused upsamples and the
    Detect head's flat outputs included) against the 128x128 tile."""
    import torch
    from vrs.synth import images, seeded_params
    desc = vrs.block(vrs.BLOCK_YOLO26, 3, nc=7, variant="n")
    x = torch.from_numpy(images(2, 64, 96)).cuda()
    outs = []
    for code in (vrs.TILE_128x128, tile):
        m = vrs.Model(ctx(), desc, 2, 64, 96, dtype, 1e-3, autotune=False)
        P = seeded_params(m.params(), seed=3, bn="random")
        stem = {i for i, (p, _, _) in enumerate(m.conv_info()) if p == "model.0"}
        w = {p[: -len(".conv.weight")] if p.endswith(".conv.weight") else p[: -len(".weight")]: v.shape
             for p, v in P.items() if v.ndim == 4}
        m.set_plan([0 if i in stem or w[p][1] == 1 else code for i, (p, _, _) in enumerate(m.conv_info())])
        m.load(P)
        outs.append([o.double().cpu() for o in m.forward(x)])
        names = m.launch_names()
    kernel = "_s32_w" if tile & 0xff == vrs.TILE_KW32 else "_s16_w"
    assert sum(kernel in s for s in names) > 70, names
    for a, b in zip(*outs):
        # float32: ~100 layers of another summation order, 1e-6 each; bfloat16:
        # roundings that flip and travel on, 0.5 % of a deep network's outputs
        rel = float((a - b).norm() / a.norm())
        assert rel < (1e-4 if dtype == vrs.F32 else 2e-2), rel


@pytest.mark.parametrize("dtype,n,c,h,w,s", [
    # LDS tile: strips of 4 rows, 64 bytes of channels, tiles of 4..40 x 10..40
    (vrs.F32, 1, 8, 1, 1, 1), (vrs.F32, 1, 24, 45, 50, 1), (vrs.F32, 2, 40, 21, 41, 2), (vrs.F32, 30, 96, 33, 37, 1),
    (vrs.BF16, 1, 8, 2, 9, 1), (vrs.BF16, 1, 40, 45, 50, 1), (vrs.BF16, 9, 136, 21, 23, 1),
    # larger ones that do not fill the row walker's bands
    (vrs.BF16, 12, 320, 33, 90, 1), (vrs.BF16, 16, 264, 41, 75, 1),
    # row walker (over 70 MB moved, bands at least 4/5 filled): 40-row bands, the last of 39 and of 1 row; 10-row bands
    (vrs.BF16, 16, 264, 79, 90, 1), (vrs.BF16, 9, 136, 281, 90, 1), (vrs.BF16, 61, 264, 29, 63, 1),
    # float32: the row walker over 512 MB moved
    (vrs.F32, 41, 264, 79, 83, 1),
])
def test_depthwise_paths(dtype, n, c, h, w, s):
    import oracle
    import torch
    from gpu_util import dev, from_nhwc, rel_err, to_nhwc
    rnd = rounder(dtype)
    rng = np.random.default_rng([n, c, h, w, s])
    x = rnd(rng.standard_normal((n, c, h, w), dtype=np.float32))
    wt = rnd((rng.standard_normal((c, 1, 3, 3)) * 0.4).astype(np.float32))
    scale = rng.uniform(0.5, 1.5, c).astype(np.float32)
    shift = rng.normal(0, 0.2, c).astype(np.float32)
    ref = oracle.affine_act(oracle.conv2d(x, wt, s, 1, c), scale, shift, 1)
    xt = to_nhwc(x, dtype, c + 8, 8)
    yt = torch.full((n, ref.shape[2], ref.shape[3], c + 8), 7.0, dtype=tdtype(dtype), device="cuda")
    ctx().conv2d(vrs.nhwc(xt, c, 8), dev(vrs.pack_conv_weight(wt, c, 1, dtype)), dev(scale), dev(shift),
                 vrs.nhwc(yt, c, 0), 3, s, c, vrs.ACT_SILU, None, dtype)
    torch.cuda.synchronize()
    err = rel_err(from_nhwc(yt, c, 0), ref, 5e-2 if dtype == vrs.F32 else 1e-1)   # bounds of the other depthwise tests
    assert err < (1e-4 if dtype == vrs.F32 else 2e-2), err
    assert torch.all(yt[..., c:] == 7.0)


@pytest.mark.parametrize("dtype,n,c,h,w,s", [
    # several images to a tile, the last one of fewer
    (vrs.F32, 9001, 64, 1, 1, 1), (vrs.F32, 701, 256, 3, 5, 1), (vrs.F32, 211, 136, 9, 7, 1), (vrs.F32, 101, 264, 14, 13, 1),
    (vrs.F32, 9001, 64, 1, 1, 2), (vrs.F32, 701, 256, 4, 3, 2), (vrs.F32, 401, 136, 7, 9, 2), (vrs.F32, 130, 264, 27, 28, 2),
    (vrs.BF16, 9001, 64, 1, 1, 1), (vrs.BF16, 701, 256, 5, 3, 1), (vrs.BF16, 211, 136, 8, 9, 1),
])
def test_depthwise_small_maps(dtype, n, c, h, w, s):
    """A period of 37 images against the oracle, the others against it bit for bit."""
    import oracle
    import torch
    from gpu_util import dev, from_nhwc, rel_err, to_nhwc
    rnd = rounder(dtype)
    rng = np.random.default_rng([n, c, h, w, s])
    x = rnd(rng.standard_normal((37, c, h, w), dtype=np.float32))
    wt = rnd((rng.standard_normal((c, 1, 3, 3)) * 0.4).astype(np.float32))
    scale = rng.uniform(0.5, 1.5, c).astype(np.float32)
    shift = rng.normal(0, 0.2, c).astype(np.float32)
    ref = oracle.affine_act(oracle.conv2d(x, wt, s, 1, c), scale, shift, 1)
    xt = to_nhwc(x, dtype, c + 8, 8)[torch.arange(n) % 37].contiguous()
    yt = torch.full((n, ref.shape[2], ref.shape[3], c + 8), 7.0, dtype=tdtype(dtype), device="cuda")
    ctx().conv2d(vrs.nhwc(xt, c, 8), dev(vrs.pack_conv_weight(wt, c, 1, dtype)), dev(scale), dev(shift),
                 vrs.nhwc(yt, c, 0), 3, s, c, vrs.ACT_SILU, None, dtype)
    torch.cuda.synchronize()
    err = rel_err(from_nhwc(yt[:37], c, 0), ref, 5e-2 if dtype == vrs.F32 else 1e-1)   # bounds of test_depthwise_paths
    assert err < (1e-4 if dtype == vrs.F32 else 2e-2), err
    assert torch.equal(yt, yt[:37][torch.arange(n) % 37]) and torch.all(yt[..., c:] == 7.0)


@pytest.mark.parametrize("dtype,b,heads,h,w", [
    (vrs.F32, 1, 1, 1, 1), (vrs.BF16, 1, 1, 1, 1),          # one key: three of the four waves have none
    (vrs.F32, 1, 2, 8, 16), (vrs.BF16, 1, 2, 8, 16),        # 128 keys: the last size shared by four waves
    (vrs.F32, 2, 1, 3, 43), (vrs.BF16, 2, 1, 3, 43),        # 129 keys: eight waves, a chunk of one key
    (vrs.F32, 1, 1, 23, 23), (vrs.BF16, 1, 1, 23, 23),      # 529 keys: a second round of chunks
    (vrs.BF16, 16, 4, 24, 24),                              # 2304 workgroups of 16 queries: the streamed kernel
    (vrs.BF16, 16, 5, 20, 20),                              # 2000: the resident kernel
    (vrs.BF16, 13, 1, 50, 50), (vrs.BF16, 11, 1, 50, 50),   # over 2048 keys: 2041 on the streamed kernel, 1727 split
])
def test_attention_paths(dtype, b, heads, h, w):
    import torch
    torch.manual_seed(b * 1000 + h * w)
    c = heads * 64
    qkv = torch.randn(b, h, w, heads * 128, device="cuda").to(tdtype(dtype))
    pe_w = (torch.randn(9, c, device="cuda") * 0.3).to(tdtype(dtype))
    pe_s, pe_t = torch.rand(c, device="cuda") + 0.5, torch.randn(c, device="cuda") * 0.1
    out = torch.full((b, h, w, c + 8), 7.0, device="cuda", dtype=tdtype(dtype))
    ctx().psa_attention(vrs.nhwc(qkv), pe_w, pe_s, pe_t, vrs.nhwc(out, c, 4), heads, dtype)
    q, k, v = qkv.double().reshape(b, h * w, heads, 128).permute(0, 2, 1, 3).split((32, 32, 64), 3)
    p = (torch.matmul(q.contiguous(), k.transpose(2, 3).contiguous()) * 32 ** -0.5).softmax(-1)
    o = torch.matmul(p, v.contiguous()).permute(0, 2, 1, 3).reshape(b, h, w, c)
    vm = torch.nn.functional.pad(v.permute(0, 2, 1, 3).reshape(b, h, w, c), (0, 0, 1, 1, 1, 1))
    pe = sum(vm[:, i // 3:i // 3 + h, i % 3:i % 3 + w] * pe_w[i].double() for i in range(9))
    ref = o + pe * pe_s.double() + pe_t.double()
    # float32: a few roundings of the largest term; bfloat16: the probabilities' and the output's 2^-9
    err = float((out[..., 4:c + 4].double() - ref).abs().max() / ref.square().mean().sqrt())
    assert err < (1e-5 if dtype == vrs.F32 else 4e-2), err
    assert torch.all(out[..., :4] == 7.0) and torch.all(out[..., c + 4:] == 7.0)


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("h,w", [(16, 16), (25, 41)])   # 256 and 1025 keys: eight waves, one and several chunks each
@pytest.mark.parametrize("lo,hi", [(0, 64), (64, 128), (192, 256), (0, 250)])
def test_attention_keys_that_score_minus_infinity(dtype, h, w, lo, hi):
    """Whole chunks of keys whose scores are -inf weigh nothing, whichever wave holds them."""
    import torch
    torch.manual_seed(h + lo)
    qkv = torch.randn(1, h, w, 128, device="cuda").to(tdtype(dtype))
    qkv[..., 0] = 1.0                                    # q's first channel
    qkv.view(1, h * w, 128)[:, lo:hi, 32] = -torch.inf   # k's first channel
    pe_w = torch.zeros(9, 64, device="cuda", dtype=tdtype(dtype))
    zero = torch.zeros(64, device="cuda")
    out = torch.zeros(1, h, w, 64, device="cuda", dtype=tdtype(dtype))
    ctx().psa_attention(vrs.nhwc(qkv), pe_w, zero, zero, vrs.nhwc(out), 1, dtype)
    q, k, v = qkv.double().reshape(h * w, 128).split((32, 32, 64), 1)
    keep = torch.ones(h * w, dtype=torch.bool, device="cuda")
    keep[lo:hi] = False
    p = (torch.matmul(q, k[keep].t().contiguous()) * 32 ** -0.5).softmax(-1)
    ref = torch.matmul(p, v[keep].contiguous()).reshape(1, h, w, 64)
    err = float((out.double() - ref).abs().max() / ref.square().mean().sqrt())
    assert err < (1e-5 if dtype == vrs.F32 else 4e-2), err   # the bounds of test_attention_paths


@pytest.mark.parametrize("h,w,nc,thr,max_det", [
    (64, 96, 5, 0.25, 10),         # 126 anchors: all kept ones sorted
    (96, 160, 80, 0.001, 300),     # 315 anchors (odd)
    (128, 128, 1, 0.0, 1024),      # one class, every anchor kept
    (640, 640, 9, 0.001, 300),     # 8400 anchors: radix select
    (1024, 1056, 3, 0.001, 1000),  # 22176 anchors: more than the registers hold
])
def test_detect_postprocess_paths(h, w, nc, thr, max_det):
    """Near-equal, saturated, underflowing, infinite and NaN logits: class,
    score and order as the plain loop over sigmoids gives them, bit for bit."""
    import torch
    rng = np.random.default_rng([h, w, nc])
    strides = (8, 16, 32)
    sizes = [(h // s) * (w // s) for s in strides]
    A, n = sum(sizes), 2
    lg = rng.normal(-3, 2, (n, nc, A)).astype(np.float32)
    kind = rng.integers(0, 12, (n, A))
    base = rng.normal(-2, 3, (n, 1, A)).astype(np.float32)
    lg = np.where((kind == 0)[:, None], base + rng.integers(0, 3, lg.shape).astype(np.float32) * np.float32(1e-7), lg)
    lg = np.where((kind == 1)[:, None], base + rng.uniform(0, 2e-3, lg.shape).astype(np.float32), lg)
    lg = np.where((kind == 2)[:, None], rng.uniform(4.9, 30, lg.shape).astype(np.float32), lg)
    lg = np.where((kind == 3)[:, None], rng.uniform(-110, -79, lg.shape).astype(np.float32), lg)
    odd = rng.choice(np.array([np.nan, np.inf, -np.inf, 0.0, -0.0], np.float32), lg.shape)
    lg = np.where((kind == 4)[:, None] & (rng.integers(0, 3, lg.shape) == 0), odd, lg).astype(np.float32)
    boxes = rng.uniform(0, 5, (n, 4, A)).astype(np.float32)

    def flat(t):   # per-scale blocks, channel-major inside each
        parts, at = [], 0
        for sz in sizes:
            parts.append(t[:, :, at:at + sz].reshape(n, -1))
            at += sz
        return torch.from_numpy(np.concatenate(parts, 1)).cuda()

    count, score, cls, anchor, xywh = ctx().detect_postprocess(flat(boxes), flat(lg), nc, h, w, strides, thr, max_det)
    p = 1.0 / (1.0 + torch.exp(-torch.from_numpy(lg).cuda()))
    best, bc = p[:, 0].clone(), torch.zeros(n, A, dtype=torch.int64, device="cuda")
    for c in range(1, nc):   # Iterator::max_by with partial_cmp().unwrap_or(Equal)
        take = ~(best > p[:, c])
        best = torch.where(take, p[:, c], best)
        bc = torch.where(take, torch.full_like(bc, c), bc)
    best, bc = best.cpu().numpy(), bc.cpu().numpy()
    for b in range(n):
        kept = np.flatnonzero(best[b] >= np.float32(thr))
        order = kept[np.argsort(-best[b][kept], kind="stable")][:max_det]
        k = int(count[b])
        assert k == len(order)
        assert np.array_equal(anchor[b, :k].cpu().numpy(), order)
        assert np.array_equal(score[b, :k].cpu().numpy().view(np.uint32), best[b][order].view(np.uint32))
        assert np.array_equal(cls[b, :k].cpu().numpy(), bc[b][order])
        assert torch.all(anchor[b, k:] == -1) and torch.all(score[b, k:] == 0) and torch.all(cls[b, k:] == -1)
        a0, want = 0, []
        for s, sz in zip(strides, sizes):
            sel = [(i, a) for i, a in enumerate(order) if a0 <= a < a0 + sz]
            for i, a in sel:
                l, t, r, bo = boxes[b, :, a]
                jx, jy = (a - a0) % (w // s), (a - a0) // (w // s)
                want.append((i, (jx + 0.5) * s + s * (r - l) * 0.5, (jy + 0.5) * s + s * (bo - t) * 0.5, s * (l + r),
                             s * (t + bo)))
            a0 += sz
        if k:
            want = np.array(sorted(want), np.float64)[:, 1:]
            assert np.max(np.abs(xywh[b, :k].cpu().numpy() - want)) < 1e-3 * 4   # float32 at up to 1100 pixels


@pytest.mark.parametrize("tile", SPLIT_TILES + [pytest.param(vrs.TILE_AUTO, id="auto")])
@pytest.mark.parametrize("n,cin,h,w,cout,k,s,res,y8", [
    (1, 64, 1, 1, 16, 1, 1, None, False),    # one pixel, half a step of K
    (1, 64, 5, 7, 48, 3, 1, "e4m3", True),   # taps of half a step
    (2, 128, 6, 5, 32, 3, 2, None, True),    # taps of one step
    (1, 192, 4, 9, 80, 1, 1, "bf16", False),
    (1, 512, 3, 3, 16, 3, 1, "bf16", True),  # deep K
])
def test_split_k_fp8(n, cin, h, w, cout, k, s, res, y8, tile):
    """The same sums in another order as the 128x128 fp8 tile (which other tests
    hold against the oracle): at most one rounding apart."""
    import torch
    torch.manual_seed(cin + cout)
    x = (torch.randn(n, h, w, cin + 16, device="cuda") * 2).to(torch.float8_e4m3fn).view(torch.uint8)
    rng = np.random.default_rng(cin)
    q, ws = vrs.pack_conv_weight_fp8((rng.standard_normal((cout, cin, k, k)) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32))
    q, sc = torch.from_numpy(q).cuda(), torch.from_numpy(ws).cuda() * (torch.rand(cout, device="cuda") + 0.5)
    sh = torch.randn(cout, device="cuda") * 0.2
    ho, wo = (h - 1) // s + 1, (w - 1) // s + 1
    rt = None
    if res:
        rt = torch.randn(n, ho, wo, cout + 16, device="cuda")
        rt = rt.to(torch.float8_e4m3fn).view(torch.uint8) if res == "e4m3" else rt.bfloat16()
    outs = []
    for t in (vrs.TILE_128x128, tile):
        y = torch.full((n, ho, wo, cout + 16), 0x55, dtype=torch.uint8, device="cuda")
        y = y if y8 else y.bfloat16()
        ctx().conv2d(vrs.nhwc(x, cin, 16), q, sc, sh, vrs.nhwc(y, cout, 16), k, s, 1, vrs.ACT_SILU,
                     None if rt is None else vrs.nhwc(rt, cout, 16), vrs.FP8, tile=t, in_scale=1.0, x_e4m3=True,
                     y_e4m3=y8, out_step=2.0 ** -5 if y8 else 0.0, res_e4m3=res == "e4m3",
                     res_step=1.0 if res == "e4m3" else 0.0)
        torch.cuda.synchronize()
        assert torch.all(y[..., :16] == 0x55)
        v = y[..., 16:].contiguous()
        outs.append((v.view(torch.float8_e4m3fn) if y8 else v).double())
    a, b = outs
    step = 2.0 ** -3 if y8 else 2.0 ** -7     # one step of the output type, relative
    small = (2.0 ** -9 if y8 else 1e-6) * float(a.abs().max())
    assert torch.all((a - b).abs() <= step * a.abs() + small)
    assert float((a != b).double().mean()) < 0.02   # float32 sums differ by 1e-6, roundings flip rarely


@pytest.mark.parametrize("points", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,q,heads,shapes", [
    (1, 1, 1, [(1, 1)]),                                      # one row of eight, one level, one pixel
    (3, 7, 5, [(9, 4), (3, 1), (2, 2)]),                      # 105 rows: the last workgroup holds one
    (2, 5, 8, [(13, 11), (7, 6), (4, 3), (2, 2)]),            # a query per workgroup
    (1, 3, 19, [(5, 4)] * 8),                                 # eight waves, queries that straddle workgroups
])
def test_msda_paths(points, n, q, heads, shapes):
    """Up to four points: a wave per level; more: the general kernel.  Points at
    infinity and NaN, and infinite weights outside the map, add nothing."""
    import oracle
    import torch
    from gpu_util import dev, rel_err
    from test_oracle_golden import msda_inputs
    value, ref, off, attw = msda_inputs(n, q, heads, 32, shapes, points)
    off[0, 0, 0, 0, 0] = (np.inf, 0.0)
    off[-1, -1, -1, -1, -1] = (np.nan, -np.inf)
    off[0, -1, -1, 0, -1] = (50.0, 0.0)
    clean = attw.copy()
    for at in ((0, 0, 0, 0, 0), (-1, -1, -1, -1, -1), (0, -1, -1, 0, -1)):
        clean[at] = 0.0
        attw[at] = np.inf
    exp = oracle.msda(value, shapes, ref, np.where(np.isfinite(off), off, 0).astype(np.float32), clean)
    out = torch.full((n * q * heads * 32 + 8,), 7.0, device="cuda")
    ctx().msda(dev(value), shapes, dev(ref), dev(off), dev(attw), out[:-8].view(n, q, heads * 32))
    torch.cuda.synchronize()
    assert rel_err(out[:-8].view(n, q, -1).cpu().numpy(), exp, 5e-2) < 1e-4   # the bound of the other float32 tests
    assert torch.all(out[-8:] == 7.0)


def test_msda_of_more_rows_than_a_launch_splits_by_level():
    """2^23 queries of 8 heads at 8 levels: 2^32 threads with a wave per level."""
    import oracle
    import torch
    from gpu_util import rel_err
    from test_oracle_golden import msda_inputs
    q, heads, shapes = 1 << 23, 8, [(2, 3)] * 8
    value, ref, off, attw = msda_inputs(1, 512, heads, 32, shapes, 1)
    exp = oracle.msda(value, shapes, ref, off, attw)
    many = [torch.from_numpy(t).cuda().repeat(1, q // 512, *[1] * (t.ndim - 2)) for t in (ref, off, attw)]
    out = torch.empty(1, q // 512, 512, heads * 32, device="cuda")
    ctx().msda(torch.from_numpy(value).cuda(), shapes, *many, out.view(1, q, heads * 32))
    assert rel_err(out[0, 0].cpu().numpy(), exp[0], 5e-2) < 1e-4   # the bound of test_msda_paths
    assert torch.equal(out, out[:, :1].expand_as(out))


@pytest.mark.parametrize("size,frames", [
    # one canvas tile of the 2x kernel and less; a pixel; a row that no dword fits
    (8, [(16, 16), (1, 1), (3, 1), (5, 16)]),
    # no frame shrinks: the three-tap kernel
    (150, [(150, 150), (61, 37), (1, 90), (149, 8)]),
    # whole tiles; exactly 2x, 4x and 8x; one pixel more (the next kernel)
    (64, [(128, 128), (256, 100), (512, 512), (129, 128), (257, 256), (513, 77)]),
    # enlarged, odd row lengths, partial tiles on both sides
    (77, [(41, 77), (77, 13), (154, 151), (301, 307), (600, 431), (77, 77)]),
    (200, [(399, 230), (7, 200), (800, 797), (1599, 1600)]),
])
def test_letterbox_paths(size, frames):
    """Frames at every byte misalignment, against the two-pass oracle bit for bit."""
    import oracle
    import torch
    rng = np.random.default_rng(size)
    offs, wh, parts, at = [], [], [], 0
    for i in range(16):
        w, h = frames[i % len(frames)]
        pad = 1 + (i - 1 - at) % 16     # the frame starts at a byte = i mod 16
        parts.append(np.full(pad, 255, np.uint8))
        at += pad
        offs.append(at)
        wh.append((w, h))
        parts.append(rng.integers(0, 256, h * w * 3, dtype=np.uint8))
        at += h * w * 3
    flat = np.concatenate(parts)
    got = ctx().letterbox(torch.from_numpy(flat).cuda(), offs, wh, size)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    for i, ((w, h), o) in enumerate(zip(wh, offs)):
        assert o % 16 == i
        ref = oracle.letterbox(flat[o:o + h * w * 3].reshape(h, w, 3), size)
        assert np.array_equal(got[i].view(np.uint32), np.asarray(ref, np.float32).reshape(got[i].shape).view(np.uint32)), (w, h, o)
