"""Single-op C ABI (include/ivh.h, ivh_conv2d_f16 ... ivh_bmm_f16) on the GPU: each entry
point runs one operation on caller-owned device buffers (torch allocations here) and is
compared with the CPU oracle on the same seeded inputs, with the op-level bar of the plan
tests (fp32 oracle: mean_rel < 2e-3, max_rel < 1e-2; data movement bit-exact).  The
padding channels of channels-last activations hold NaN bit patterns, so a kernel that lets
them reach an output fails."""
import time

import numpy as np
import pytest
import torch

import infvino_amd as ia
import infvino_amd.ops as ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

F32_MEAN, F32_MAX = 2e-3, 1e-2
NAN16 = 0x7E00


def _dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a, np.uint16).view(np.int16).copy()).to("cuda")


def _host(t: torch.Tensor) -> np.ndarray:
    torch.cuda.synchronize()
    return t.cpu().numpy().view(np.uint16)


def _nhwc(x: np.ndarray, B, C, H, W, fill=NAN16) -> np.ndarray:
    cs = (C + 7) // 8 * 8
    out = np.full((B, H, W, cs), fill, np.uint16)
    out[..., :C] = x.reshape(B, C, H, W).transpose(0, 2, 3, 1)
    return out


def _from_nhwc(y: np.ndarray, B, C, H, W) -> np.ndarray:
    cs = (C + 7) // 8 * 8
    return y.reshape(B, H, W, cs)[..., :C].transpose(0, 3, 1, 2).reshape(B, -1)


def _ok(got, ref, label):
    mean_rel, max_rel, max_abs, _ = O.rel_errors(O.h2f(got.ravel()), O.h2f(ref.ravel()))
    print(f"{label}: mean_rel={mean_rel:.2e} max_rel={max_rel:.2e} max_abs={max_abs:.2e}")
    return mean_rel < F32_MEAN and max_rel < F32_MAX


def _pack(d, w, b):
    packed = torch.empty(ops.conv_packed_bytes(d), dtype=torch.uint8, device="cuda")
    ops.pack_conv_weights(d, w, b, packed.data_ptr())
    return packed


CONVS = [
    # cin, cout, h, w, k, s, p, g, act, channels_last, residual
    (64, 128, 20, 20, 1, 1, 0, 1, ops.ACT_SILU, 1, False),     # 1x1 implicit GEMM
    (24, 40, 17, 19, 3, 1, 1, 1, ops.ACT_HSWISH, 1, True),     # 3x3 s1 LDS patch, ragged, residual
    (21, 32, 15, 15, 3, 2, 1, 1, ops.ACT_SILU, 1, False),      # 3x3 s2 im2col, Cin % 8 != 0
    (8, 20, 9, 11, 5, 1, 2, 1, ops.ACT_SIGMOID, 1, True),      # 5x5, 8 channels a piece, residual
    (13, 48, 17, 14, 3, 2, 1, 1, ops.ACT_SILU, 1, True),       # 3x3 s2 LDS patch, pad channels, residual
    (128, 256, 10, 10, 3, 1, 1, 1, ops.ACT_RELU, 1, False),    # wide, K step 64
    (3, 16, 64, 64, 3, 2, 1, 1, ops.ACT_SILU, 0, False),       # stem, planar in and out
    (16, 1, 4, 64, 1, 1, 0, 1, ops.ACT_NONE, 0, False),        # planar 1x1, one output channel
    (32, 64, 10, 10, 3, 1, 1, 4, ops.ACT_RELU, 1, False),      # grouped, direct kernel
    (48, 48, 14, 14, 5, 2, 2, 48, ops.ACT_HSWISH, 1, True),    # depthwise 5x5 s2, residual
]


@pytest.mark.parametrize("cin,cout,h,w,k,s,p,g,act,cl,res", CONVS,
                         ids=[f"{c[0]}-{c[1]}-{c[2]}x{c[3]}-k{c[4]}s{c[5]}g{c[7]}-cl{c[9]}" for c in CONVS])
def test_abi_conv2d(cin, cout, h, w, k, s, p, g, act, cl, res):
    B = 3
    rng = np.random.default_rng(cin * 1000 + cout)
    d = ops.conv_desc(cin, cout, h, w, k, s, p, g, act, True, cl)
    ho, wo = ops.conv_out_dims(d)
    assert (ho, wo) == ((h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1)
    x = O.f2h(rng.random(B * cin * h * w).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * (cin // g) * k * k) * np.sqrt(2.0 / (cin // g * k * k))).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.01).astype(np.float32))
    r = O.f2h(rng.random(B * cout * ho * wo).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    conv = ops.dwconv if g == cin == cout and k in (3, 5) else ops.conv2d
    if cl:
        xd = _dev(_nhwc(x, B, cin, h, w))
        yd = _dev(np.full(B * ho * wo * ((cout + 7) // 8 * 8), NAN16, np.uint16))
        rd = _dev(_nhwc(r, B, cout, ho, wo)) if res else None
    else:
        xd, yd = _dev(x), _dev(np.full(B * cout * ho * wo, NAN16, np.uint16))
        rd = _dev(r) if res else None
    conv(d, xd.data_ptr(), packed.data_ptr(), rd.data_ptr() if rd is not None else None, yd.data_ptr(), B)
    y = _host(yd)
    got = _from_nhwc(y, B, cout, ho, wo) if cl else y.reshape(B, -1)
    for b in range(B):
        ref = O.conv2d(x[b * cin * h * w:(b + 1) * cin * h * w], wt, bias,
                       None if r is None else r[b * cout * ho * wo:(b + 1) * cout * ho * wo],
                       cin, h, w, cout, k, s, p, g, ho, wo, act, O.F32, 2)
        assert _ok(got[b], ref, f"conv {cin}->{cout} {h}x{w} k{k} s{s} g{g} cl{cl} image {b}")


def test_abi_dwconv_rejects_dense():
    d = ops.conv_desc(16, 16, 8, 8, 3, 1, 1, 1)
    with pytest.raises(RuntimeError, match="depthwise"):
        ops.dwconv(d, 16, 16, None, 16, 1)   # rejected before any pointer is used


@pytest.mark.parametrize("n_in,n_out,act", [(576, 1024, ops.ACT_HSWISH), (100, 37, ops.ACT_SIGMOID)])
def test_abi_gemv(n_in, n_out, act):
    B = 5
    rng = np.random.default_rng(n_in)
    d = ops.conv_desc(n_in, n_out, 1, 1, act=act, has_bias=True, channels_last=False)
    x = O.f2h(rng.random(B * n_in).astype(np.float32))
    wt = O.f2h((rng.standard_normal(n_out * n_in) * np.sqrt(2.0 / n_in)).astype(np.float32))
    bias = O.f2h((rng.standard_normal(n_out) * 0.01).astype(np.float32))
    packed = _pack(d, wt, bias)
    xd, yd = _dev(x), _dev(np.zeros(B * n_out, np.uint16))
    ops.gemv(d, xd.data_ptr(), packed.data_ptr(), yd.data_ptr(), B)
    y = _host(yd).reshape(B, n_out)
    for b in range(B):
        ref = O.conv2d(x[b * n_in:(b + 1) * n_in], wt, bias, None, n_in, 1, 1, n_out, 1, 1, 0, 1, 1, 1, act, O.F32, 1)
        assert _ok(y[b], ref, f"gemv {n_in}->{n_out} image {b}")


@pytest.mark.parametrize("n_in,n_out,res,pad", [(64, 10, False, 0), (576, 1000, True, 0), (100, 37, True, 0),
                                                (16, 24, False, 1)])
def test_abi_conv2d_one_pixel_planes(n_in, n_out, res, pad):
    """ivh_conv2d_f16 on planes of one pixel (a squeeze-and-excite layer's 1x1 conv) reads the
    packing that the descriptor got."""
    B = 5
    rng = np.random.default_rng(n_in)
    d = ops.conv_desc(n_in, n_out, 1, 1, 1, 1, pad, act=ops.ACT_HSIGMOID, channels_last=False)
    ho, wo = ops.conv_out_dims(d)
    no = n_out * ho * wo
    x = O.f2h(rng.random(B * n_in).astype(np.float32))
    wt = O.f2h((rng.standard_normal(n_out * n_in) * np.sqrt(2.0 / n_in)).astype(np.float32))
    bias = O.f2h((rng.standard_normal(n_out) * 0.01).astype(np.float32))
    r = O.f2h(rng.random(B * no).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    xd, yd, rd = _dev(x), _dev(np.full(B * no + 8, NAN16, np.uint16)), _dev(r) if res else None
    ops.conv2d(d, xd.data_ptr(), packed.data_ptr(), rd.data_ptr() if res else None, yd.data_ptr(), B)
    y = _host(yd)
    assert np.all(y[B * no:] == NAN16)
    for b in range(B):
        ref = O.conv2d(x[b * n_in:(b + 1) * n_in], wt, bias, None if r is None else r[b * no:(b + 1) * no], n_in, 1, 1,
                       n_out, 1, 1, pad, 1, ho, wo, ops.ACT_HSIGMOID, O.F32, 1 if pad == 0 else 0)
        assert _ok(y[b * no:(b + 1) * no], ref, f"one pixel {n_in}->{n_out} image {b}")


def test_abi_eltwise():
    B, n = 2, 4000
    rng = np.random.default_rng(7)
    a = O.f2h((rng.random(B * n) * 4 - 2).astype(np.float32))
    bv = O.f2h((rng.random(B * n) + 0.5).astype(np.float32))
    L = O.lib()
    ad, bd, yd = _dev(a), _dev(bv), _dev(np.zeros(B * n, np.uint16))
    for op in range(4):
        ops.eltwise(op, ad.data_ptr(), bd.data_ptr(), yd.data_ptr(), n, B)
        ref = np.empty(B * n, np.uint16)
        L.ivo_ew_binary(a, bv, ref, B * n, op, 0)
        assert np.array_equal(_host(yd), ref), f"binary op {op}"
    ops.eltwise(2, ad.data_ptr(), bd.data_ptr(), yd.data_ptr(), n, B, b_scalar=True)
    ref = O.f2h(O.h2f(a) * O.h2f(bv[:1]))
    assert np.array_equal(_host(yd), ref), "scalar multiply"
    # unary: canonical activation codes, against the formulas in fp32 with one rounding
    af = O.h2f(a).astype(np.float32)
    forms = {ops.ACT_SILU: af / (1 + np.exp(-af)), ops.ACT_RELU: np.maximum(af, 0),
             ops.ACT_HSWISH: af * np.clip(af + 3, 0, 6) / 6, ops.ACT_HSIGMOID: np.clip(af + 3, 0, 6) / 6,
             ops.ACT_SIGMOID: 1 / (1 + np.exp(-af))}
    for act, f in forms.items():
        ops.eltwise(act, ad.data_ptr(), None, yd.data_ptr(), n, B)
        got = O.h2f(_host(yd))
        ref = O.h2f(O.f2h(f.astype(np.float32)))
        assert np.max(np.abs(got - ref)) <= 2e-3 * max(1.0, float(np.max(np.abs(ref)))), f"unary {act}"


def test_abi_pool_softmax_bmm():
    rng = np.random.default_rng(9)
    L = O.lib()
    B, C, H, W = 2, 16, 20, 20
    x = O.f2h((rng.random(B * C * H * W) * 2 - 1).astype(np.float32))
    xd = _dev(x)
    # maxpool 5/1/2 (SPPF) and 3/2/1: bit-exact
    for k, s, p in [(5, 1, 2), (3, 2, 1)]:
        ho, wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
        yd = _dev(np.zeros(B * C * ho * wo, np.uint16))
        ops.pool(ops.POOL_MAX, xd.data_ptr(), yd.data_ptr(), C, H, W, k, s, p, B)
        y = _host(yd).reshape(B, -1)
        for b in range(B):
            ref = np.empty(C * ho * wo, np.uint16)
            L.ivo_maxpool(x[b * C * H * W:(b + 1) * C * H * W], ref, C, H, W, ho, wo, k, s, p)
            assert np.array_equal(y[b], ref), f"maxpool {k}/{s}/{p}"
    yd = _dev(np.zeros(B * C * H * W * 4, np.uint16))
    ops.pool(ops.POOL_RESIZE, xd.data_ptr(), yd.data_ptr(), C, H, W, 0, 2, 0, B)
    y = _host(yd).reshape(B, -1)
    for b in range(B):
        ref = np.empty(C * H * W * 4, np.uint16)
        L.ivo_resize_nn(x[b * C * H * W:(b + 1) * C * H * W], ref, C, H, W, 2)
        assert np.array_equal(y[b], ref), "resize x2"
    # softmax over a strided axis (vector path) and over the last axis
    for outer, axis, inner in [(4, 16, 8400 // 4), (3, 10, 1), (2, 24, 20)]:
        n = outer * axis * inner
        s = O.f2h((rng.standard_normal(B * n) * 3).astype(np.float32))
        sd, od = _dev(s), _dev(np.zeros(B * n, np.uint16))
        ops.softmax(sd.data_ptr(), od.data_ptr(), outer, axis, inner, B)
        got = _host(od).reshape(B, -1)
        for b in range(B):
            ref = np.empty(n, np.uint16)
            L.ivo_softmax_axis(s[b * n:(b + 1) * n], ref, outer, axis, inner)
            assert _ok(got[b], ref, f"softmax {outer}x{axis}x{inner}")
    # batched matmul (the C2PSA attention shapes, scaled down)
    bb, m, k, n = 2, 40, 32, 48
    a = O.f2h((rng.standard_normal(B * bb * m * k) * 0.5).astype(np.float32))
    bm = O.f2h((rng.standard_normal(B * bb * k * n) * 0.5).astype(np.float32))
    ad, bd, yd = _dev(a), _dev(bm), _dev(np.zeros(B * bb * m * n, np.uint16))
    ops.bmm(ad.data_ptr(), bd.data_ptr(), yd.data_ptr(), bb, m, k, n, B)
    got = _host(yd).reshape(B, -1)
    for b in range(B):
        ref = np.empty(bb * m * n, np.uint16)
        L.ivo_bmm(a[b * bb * m * k:(b + 1) * bb * m * k], bm[b * bb * k * n:(b + 1) * bb * k * n], ref, bb, m, k, n)
        assert _ok(got[b], ref, "bmm")


@pytest.mark.parametrize("k,c,h,w,batch,off", [
    (5, 128, 20, 20, 3, 0),    # five planes a work-group, the last group partial
    (5, 3, 1, 1, 1, 0),        # the smallest plane
    (5, 7, 13, 17, 2, 0),      # odd width: single-element loads and stores
    (5, 6, 9, 10, 2, 1),       # even width at an odd element offset
    (3, 5, 4, 6, 2, 0),        # three-wide windows, one register block of rows
    (3, 2, 5, 3, 1, 0),
    (5, 2, 200, 160, 1, 0),    # two bands of rows per plane
    (5, 2, 300, 160, 1, 0),    # three: a band with halo rows on both sides
    (3, 3, 331, 158, 2, 0),    # the same three rows wide, the last band shorter
    (5, 1, 9, 4001, 1, 0),     # rows so wide that a band is one register block
    (3, 1, 6, 9000, 1, 0),     # wider than a band: the scalar kernel
])
def test_abi_maxpool_planes(k, c, h, w, batch, off):
    """Stride-1 same-size max pools on planes, with infinities and NaNs among the values:
    bit for bit the fmaxf chain from below every fp16 value (NaN taps ignored)."""
    rng = np.random.default_rng(k * 1000 + w)
    x = rng.standard_normal((batch, c, h, w)).astype(np.float16)
    for v in (np.inf, -np.inf, np.nan):
        x[rng.random(x.shape) < 0.02] = v
    x.reshape(-1)[: min(x.size, 40)] = np.nan  # a window of nothing but NaN
    p = k // 2
    z = np.pad(np.where(np.isnan(x), np.float16(-np.inf), x), ((0, 0), (0, 0), (p, p), (p, p)),
               constant_values=-np.inf)
    ref = np.full_like(x, -np.inf)
    for i in range(k):
        for j in range(k):
            ref = np.maximum(ref, z[:, :, i:i + h, j:j + w])
    xd = torch.zeros(x.size + 8, dtype=torch.float16, device="cuda")
    yd = torch.full((x.size + 8,), 7.0, dtype=torch.float16, device="cuda")
    xd[off:off + x.size] = torch.from_numpy(x.reshape(-1)).cuda()
    ops.pool(ops.POOL_MAX, xd[off:].data_ptr(), yd[off:].data_ptr(), c, h, w, k, 1, p, batch)
    y = yd.cpu().numpy()
    assert np.array_equal(y[off:off + x.size].reshape(x.shape), ref)
    assert np.all(y[:off] == 7.0) and np.all(y[off + x.size:] == 7.0)


def test_abi_maxpool_more_planes_than_a_grid_dimension():
    """2^24 and some planes, one to a work-group (17 GB in and out): the first and last ones, and
    those on either side of the slices' border."""
    batch, c, w = 65535, 257, 257
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 17 GB of free memory")
    x = torch.empty(batch, c * w, dtype=torch.float16, device="cuda")
    x[:] = ((torch.arange(c * w, device="cuda") * 7919) % 10007 - 5000).half()
    x[:, 0] = (torch.arange(batch, device="cuda") % 2048).half()  # images differ
    y = torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    ops.pool(ops.POOL_MAX, x.data_ptr(), y.data_ptr(), c, 1, w, 3, 1, 1, batch)
    torch.cuda.synchronize()
    edge = (((1 << 24) - 1) // c)  # images a launch holds
    for i in (0, 1, edge - 1, edge, edge + 1, batch - 1):
        p = torch.nn.functional.pad(x[i].view(c, w).float(), (1, 1), value=float("-inf"))
        ref = torch.maximum(torch.maximum(p[:, :-2], p[:, 1:-1]), p[:, 2:])
        assert torch.equal(y[i].view(c, w).float(), ref), f"image {i}"
    assert not torch.isnan(y[:, ::1001]).any()
    del x, y, p, ref
    torch.cuda.empty_cache()


@pytest.mark.parametrize("cin,cout,h,w,res,off", [
    (9, 9, 2, 4, False, 0),       # the fewest pixels and channels of the MFMA route
    (64, 128, 8, 8, False, 0),    # planar streaming kernel
    (130, 140, 4, 10, True, 0),   # planar implicit GEMM: a K remainder, two channel tiles, residual
    (24, 33, 6, 20, True, 1),     # pointers one element off a 16-byte boundary: the direct kernel
    (24, 8, 6, 20, False, 0),     # up to 8 output channels, and ...
    (24, 33, 5, 5, False, 0),     # ... planes of an odd size: the direct family
    (2, 130, 8, 8, True, 0),      # a few input channels: the direct kernel, here on few pixels, ...
    (3, 9, 192, 200, False, 0),   # ... here with few outputs of many
    (3, 40, 8, 8, False, 0),      # few input channels on the planar streaming kernel
])
def test_abi_pointwise_planes(cin, cout, h, w, res, off):
    B, n_in, n_out = 3, cin * h * w, cout * h * w
    rng = np.random.default_rng(cin + cout)
    d = ops.conv_desc(cin, cout, h, w, act=ops.ACT_SILU, channels_last=False)
    x = O.f2h(rng.random(B * n_in).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * cin) * np.sqrt(2.0 / cin)).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.01).astype(np.float32))
    r = O.f2h(rng.random(B * n_out).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    pad = lambda a: _dev(np.concatenate([np.full(off, NAN16, np.uint16), a, np.full(8, NAN16, np.uint16)]))
    xd, yd, rd = pad(x), pad(np.full(B * n_out, NAN16, np.uint16)), pad(r) if res else None
    ops.conv2d(d, xd[off:].data_ptr(), packed.data_ptr(), rd[off:].data_ptr() if res else None, yd[off:].data_ptr(), B)
    y = _host(yd)
    assert np.all(y[:off] == NAN16) and np.all(y[off + B * n_out:] == NAN16)
    got = y[off:off + B * n_out].reshape(B, -1)
    for b in range(B):
        ref = O.conv2d(x[b * n_in:(b + 1) * n_in], wt, bias, None if r is None else r[b * n_out:(b + 1) * n_out],
                       cin, h, w, cout, 1, 1, 0, 1, h, w, ops.ACT_SILU, O.F32, 2)
        assert _ok(got[b], ref, f"planes {cin}->{cout} image {b}")


@pytest.mark.parametrize("cin,cout,h,w,B,act", [
    (8, 3, 64, 64, 15, ops.ACT_NONE), (16, 13, 59, 59, 15, ops.ACT_SILU), (51, 19, 90, 90, 14, ops.ACT_HSWISH),
    (13, 41, 71, 71, 12, ops.ACT_RELU), (126, 63, 92, 93, 32, ops.ACT_SILU), (90, 101, 46, 47, 28, ops.ACT_SILU),
])
def test_abi_pointwise_ragged_outputs(cin, cout, h, w, B, act):
    """Channels-last 1x1 convs of many pixels (the streaming kernel) whose output channels leave a
    partial last piece: its values one by one, and the pixel's padding untouched."""
    rng = np.random.default_rng(cin + cout)
    d = ops.conv_desc(cin, cout, h, w, act=act)
    x = O.f2h((rng.random(B * cin * h * w) * 2 - 1).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * cin) * np.sqrt(2.0 / cin)).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.5).astype(np.float32))
    packed, c8 = _pack(d, wt, bias), (cout + 7) // 8 * 8
    xd, yd = _dev(_nhwc(x, B, cin, h, w)), _dev(np.full(B * h * w * c8 + 16, 0x1234, np.uint16))
    ops.conv2d(d, xd.data_ptr(), packed.data_ptr(), None, yd.data_ptr(), B)
    y = _host(yd)
    assert np.all(y[-16:] == 0x1234) and np.all(y[:-16].reshape(-1, c8)[:, cout:] == 0x1234)
    got = _from_nhwc(y[:-16], B, cout, h, w)
    for b in (0, B - 1):
        ref = O.conv2d(x[b * cin * h * w:(b + 1) * cin * h * w], wt, bias, None, cin, h, w, cout, 1, 1, 0, 1, h, w, act,
                       O.F32, 2)
        assert _ok(got[b], ref, f"streaming 1x1 {cin}->{cout} image {b}")


@pytest.mark.parametrize("cin,cout,h,w,k,s,B,res", [
    (256, 256, 20, 20, 3, 1, 1, False),   # 32 x 32 tiles, eight waves of nine chunks
    (128, 100, 13, 11, 3, 2, 2, True),    # the same with uneven K shares, ragged channels, residual
    (40, 33, 7, 9, 1, 1, 1, False),       # 32 x 32 tiles, four waves, the last ones without work
    (21, 19, 5, 5, 3, 1, 1, True),        # Cin % 8: chunks of four pieces straddle taps, masked tails
    (8, 12, 6, 6, 5, 1, 3, False),        # four taps a chunk
    (128, 192, 40, 40, 3, 1, 1, True),    # 64 x 32 tiles, eight waves
    (64, 64, 40, 40, 3, 1, 8, True),      # 64 x 64 tiles, pixels of two images in a tile
    (124, 130, 39, 39, 1, 1, 3, False),   # the same with a nearly empty last channel tile, Cin % 8
    (60, 130, 39, 39, 1, 1, 3, False),    # two chunks of channels: the implicit GEMM
    (256, 192, 25, 25, 1, 1, 3, True),    # 32 x 32 tiles, two chunks a wave, a partial last pixel tile
    (256, 64, 3, 3, 1, 2, 5, False),      # stride 2 pointwise
])
def test_abi_small_grid_conv(cin, cout, h, w, k, s, B, res):
    """Convs of few pixels (K split over a work-group's waves) at the edges of its tiles."""
    p, act = k // 2, ops.ACT_SILU
    rng = np.random.default_rng(cin * 7 + cout)
    d = ops.conv_desc(cin, cout, h, w, k, s, p, act=act)
    ho, wo = ops.conv_out_dims(d)
    x = O.f2h((rng.random(B * cin * h * w) * 2 - 1).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * cin * k * k) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.1).astype(np.float32))
    r = O.f2h(rng.random(B * cout * ho * wo).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    xd, rd = _dev(_nhwc(x, B, cin, h, w)), _dev(_nhwc(r, B, cout, ho, wo)) if res else None
    yd = _dev(np.full(B * ho * wo * ((cout + 7) // 8 * 8) + 64, NAN16, np.uint16))
    ops.conv2d(d, xd.data_ptr(), packed.data_ptr(), rd.data_ptr() if res else None, yd.data_ptr(), B)
    y = _host(yd)
    assert np.all(y[-64:] == NAN16)
    got = _from_nhwc(y[:-64], B, cout, ho, wo)
    for b in range(B):
        ref = O.conv2d(x[b * cin * h * w:(b + 1) * cin * h * w], wt, bias,
                       None if r is None else r[b * cout * ho * wo:(b + 1) * cout * ho * wo],
                       cin, h, w, cout, k, s, p, 1, ho, wo, act, O.F32, 2)
        assert _ok(got[b], ref, f"small-grid conv {cin}->{cout} k{k} s{s} image {b}")


@pytest.mark.parametrize("bb,m,k,n,batch", [
    (1, 1, 1, 1, 1), (2, 65, 63, 129, 2), (3, 49, 64, 49, 1), (1, 130, 70, 64, 3), (2, 33, 201, 17, 2),
    (1, 128, 128, 128, 1), (2, 8, 65, 65, 5),
])
def test_abi_bmm_edges(bb, m, k, n, batch):
    """Both tile shapes (N up to 64 and above) at odd row lengths, K remainders and partial tiles."""
    rng = np.random.default_rng(m * n + k)
    L = O.lib()
    a = O.f2h((rng.standard_normal(batch * bb * m * k) * 0.5).astype(np.float32))
    bm = O.f2h((rng.standard_normal(batch * bb * k * n) * 0.5).astype(np.float32))
    ad, bd = _dev(a), _dev(bm)
    yd = _dev(np.full(batch * bb * m * n + 16, NAN16, np.uint16))
    ops.bmm(ad.data_ptr(), bd.data_ptr(), yd.data_ptr(), bb, m, k, n, batch)
    y = _host(yd)
    assert np.all(y[-16:] == NAN16)
    got = y[:-16].reshape(batch, -1)
    for b in range(batch):
        ref = np.empty(bb * m * n, np.uint16)
        L.ivo_bmm(a[b * bb * m * k:(b + 1) * bb * m * k], bm[b * bb * k * n:(b + 1) * bb * k * n], ref, bb, m, k, n)
        assert _ok(got[b], ref, f"bmm {bb}x{m}x{k}x{n} image {b}")


@pytest.mark.parametrize("bb,batch", [((1 << 18) + 1, 64), ((1 << 24) + 5, 2)])
def test_abi_bmm_more_tiles_than_a_grid_dimension(bb, batch):
    """2^24 and some matrices of one value: their tiles exceed one dimension of a launch, over
    the images or within one."""
    a = (torch.arange(bb * batch, device="cuda") % 61).half()
    b = (torch.arange(bb * batch, device="cuda") % 29 - 14).half()
    y = torch.full((bb * batch,), float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    ops.bmm(a.data_ptr(), b.data_ptr(), y.data_ptr(), bb, 1, 1, 1, batch)
    torch.cuda.synchronize()
    assert torch.equal(y, a * b)


@pytest.mark.parametrize("axis", [1, 7, 8, 63, 64, 65, 128, 129, 256, 399, 512, 513, 1024, 2047, 2048, 2049])
def test_abi_softmax_rows(axis):
    """Rows of every lane count and piece count, at odd offsets, with a masked (-inf), a lowest
    (-65504), an all-equal and a large row."""
    rng = np.random.default_rng(axis)
    L, outer = O.lib(), 37
    v = (rng.standard_normal((outer, axis)) * 3).astype(np.float32)
    v[1, : axis // 2] = -np.inf
    v[2, axis // 3:] = -65504
    v[3] = 65504
    v[4] = -65504
    s = O.f2h(v.ravel())
    sd = torch.zeros(s.size + 1, dtype=torch.int16, device="cuda")
    sd[1:] = _dev(s)
    od = _dev(np.full(s.size + 17, NAN16, np.uint16))
    ops.softmax(sd[1:].data_ptr(), od[1:].data_ptr(), outer, axis, 1, 1)
    y = _host(od)
    assert y[0] == NAN16 and np.all(y[1 + s.size:] == NAN16)
    ref = np.empty(s.size, np.uint16)
    L.ivo_softmax_axis(s, ref, outer, axis, 1)
    assert _ok(y[1:1 + s.size], ref, f"softmax rows of {axis}")


@pytest.mark.parametrize("cin,cout,h,w,k,s,B,res", [
    (256, 128, 40, 40, 1, 1, 8, True),    # K halves of four steps, 128-channel tiles, residual
    (72, 200, 29, 31, 3, 2, 40, False),   # an odd step count over the halves, partial tiles both ways
    (64, 64, 80, 80, 3, 2, 11, False),    # 64-channel tiles, K halves with taps
    (64, 64, 80, 80, 3, 2, 8, False),     # ... and a batch that the small-grid kernel takes
    (264, 40, 33, 35, 1, 1, 20, True),    # the same, 9 steps, 40 of 64 channels
    (40, 256, 53, 53, 1, 1, 7, False),    # whole K: two steps, the second ragged
    (32, 136, 61, 59, 3, 2, 40, True),    # whole K with taps, a second channel tile of 8
    (192, 128, 64, 64, 1, 1, 16, False),  # streamed pixels: four blocks a work-group
    (136, 72, 81, 83, 1, 1, 11, False),   # a chunk of 8 channels, 8 of a wave's channels, a last block of 17 pixels
    (384, 104, 90, 91, 1, 1, 13, False),  # six chunks, uneven shares
])
def test_abi_dma_implicit_gemm(cin, cout, h, w, k, s, B, res):
    """Implicit-GEMM convs through the DMA-fed kernel: image 0 and the last one against the oracle,
    and every image equal to the same image at another place of the batch."""
    p, act = k // 2, ops.ACT_SILU
    rng = np.random.default_rng(cin * 7 + cout)
    d = ops.conv_desc(cin, cout, h, w, k, s, p, act=act)
    ho, wo = ops.conv_out_dims(d)
    x = O.f2h((rng.random(B * cin * h * w) * 2 - 1).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * cin * k * k) * np.sqrt(2.0 / (cin * k * k))).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.1).astype(np.float32))
    r = O.f2h(rng.random(B * cout * ho * wo).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    n = B * ho * wo * cout

    def run(shift):
        roll = lambda a: None if a is None else np.roll(a.reshape(B, -1), shift, axis=0).ravel()
        xd, rd = _dev(_nhwc(roll(x), B, cin, h, w)), _dev(_nhwc(roll(r), B, cout, ho, wo)) if res else None
        yd = _dev(np.full(n + 64, NAN16, np.uint16))
        ops.conv2d(d, xd.data_ptr(), packed.data_ptr(), rd.data_ptr() if res else None, yd.data_ptr(), B)
        y = _host(yd)
        assert np.all(y[n:] == NAN16)
        return np.roll(_from_nhwc(y[:n], B, cout, ho, wo), -shift, axis=0)

    got = run(0)
    assert np.array_equal(got, run(3))
    for b in (0, B - 1):
        ref = O.conv2d(x[b * cin * h * w:(b + 1) * cin * h * w], wt, bias,
                       None if r is None else r[b * cout * ho * wo:(b + 1) * cout * ho * wo],
                       cin, h, w, cout, k, s, p, 1, ho, wo, act, O.F32, 2)
        assert _ok(got[b], ref, f"DMA implicit GEMM {cin}->{cout} k{k} s{s} image {b}")


@pytest.mark.parametrize("c,h,w,k,s,B,res", [
    (2, 5, 5, 3, 1, 2, False), (7, 9, 11, 5, 2, 1, True), (9, 14, 14, 3, 2, 3, False), (51, 20, 20, 3, 1, 4, True),
    (145, 13, 17, 5, 1, 2, False), (70, 28, 28, 5, 2, 256, False), (33, 112, 112, 3, 1, 2, False),
    (325, 20, 20, 5, 1, 2, True),    # 41 groups, a prime: tiles of one group
    (328, 13, 9, 5, 1, 3, False),    # the same without a partial group
    (147, 160, 160, 3, 1, 1, True),  # 19 groups on rows of 160 pixels: two columns a tile
    (65, 3, 116600, 3, 1, 1, False),  # rows of more than 2^24 bytes: the any-layout kernel
])
def test_abi_depthwise_ragged_channels(c, h, w, k, s, B, res):
    """Depthwise convs whose channel count leaves a partial last piece (tile and strip kernels):
    NaN in the padding channels reaches no output, and the output's own padding stays."""
    p, act = k // 2, ops.ACT_HSWISH
    rng = np.random.default_rng(c * 10 + k)
    d = ops.conv_desc(c, c, h, w, k, s, p, c, act)
    ho, wo = ops.conv_out_dims(d)
    x = O.f2h((rng.random(B * c * h * w) * 2 - 1).astype(np.float32))
    wt = O.f2h((rng.standard_normal(c * k * k) * np.sqrt(2.0 / (k * k))).astype(np.float32))
    bias = O.f2h((rng.standard_normal(c) * 0.1).astype(np.float32))
    r = O.f2h(rng.random(B * c * ho * wo).astype(np.float32)) if res else None
    packed = _pack(d, wt, bias)
    xd, rd = _dev(_nhwc(x, B, c, h, w)), _dev(_nhwc(r, B, c, ho, wo)) if res else None
    c8 = (c + 7) // 8 * 8
    yd = _dev(np.full(B * ho * wo * c8 + 16, 0x1234, np.uint16))
    ops.dwconv(d, xd.data_ptr(), packed.data_ptr(), rd.data_ptr() if res else None, yd.data_ptr(), B)
    y = _host(yd)
    assert np.all(y[-16:] == 0x1234) and np.all(y[:-16].reshape(-1, c8)[:, c:] == 0x1234)
    got = _from_nhwc(y[:-16], B, c, ho, wo)
    for b in (0, B - 1):
        ref = O.conv2d(x[b * c * h * w:(b + 1) * c * h * w], wt, bias,
                       None if r is None else r[b * c * ho * wo:(b + 1) * c * ho * wo],
                       c, h, w, c, k, s, p, c, ho, wo, act, O.F32, 2)
        assert _ok(got[b], ref, f"depthwise {c} k{k} s{s} image {b}")


@pytest.mark.parametrize("cin,cout,h,w,B,act", [
    (3, 16, 64, 64, 2, ops.ACT_SILU),    # whole 16-pixel blocks, 8-byte stores
    (3, 16, 28, 28, 3, ops.ACT_HSWISH),  # width a multiple of 4: 8-byte pieces, rows of 14 outputs
    (3, 9, 33, 40, 1, ops.ACT_RELU),     # odd height, ragged channels
    (2, 16, 6, 12, 2, ops.ACT_NONE),     # fewer pixels than a block, rows of 6
    (1, 1, 5, 4, 1, ops.ACT_SILU),
    (3, 16, 8, 816, 1, ops.ACT_SILU),    # the widest staged rows of 4-pixel pieces
    (3, 16, 8, 820, 1, ops.ACT_SILU),    # ... and wider: the general kernel
])
def test_abi_stem_planes(cin, cout, h, w, B, act):
    """The 3x3 stride-2 stem from planes to planes."""
    rng = np.random.default_rng(w)
    d = ops.conv_desc(cin, cout, h, w, 3, 2, 1, act=act, channels_last=False)
    ho, wo = ops.conv_out_dims(d)
    x = O.f2h((rng.random(B * cin * h * w) * 2 - 1).astype(np.float32))
    wt = O.f2h((rng.standard_normal(cout * cin * 9) * np.sqrt(2.0 / (cin * 9))).astype(np.float32))
    bias = O.f2h((rng.standard_normal(cout) * 0.1).astype(np.float32))
    packed = _pack(d, wt, bias)
    n = B * cout * ho * wo
    xd, yd = _dev(x), _dev(np.full(n + 16, NAN16, np.uint16))
    ops.conv2d(d, xd.data_ptr(), packed.data_ptr(), None, yd.data_ptr(), B)
    y = _host(yd)
    assert np.all(y[n:] == NAN16)
    got = y[:n].reshape(B, -1)
    for b in range(B):
        ref = O.conv2d(x[b * cin * h * w:(b + 1) * cin * h * w], wt, bias, None, cin, h, w, cout, 3, 2, 1, 1, ho, wo,
                       act, O.F32, 0)
        assert _ok(got[b], ref, f"stem {cin}->{cout} {h}x{w} image {b}")


def test_readback_into_pinned_memory(tmp_path):
    """A pinned destination: the same values, and, as one copy without the ring's detour, no
    slower than the same read into pageable memory.  A device destination is the runtime's
    business too: written or refused, never touched by the host."""
    hw, batch = 1024, 8
    n = hw * hw
    path = tmp_path / "io.plan"
    path.write_text(f"input x 1 1 {hw} {hw}\ntensor y 1 1 {hw} {hw}\nnode copy_c x y HW={n} c0=0 cnt=1 dst_off=0\noutput y\n")
    m = ia.PlanModel(str(path), 0, batch, ia.IVH_FLAG_NO_FUSE)
    x = np.resize(np.arange(65536, dtype=np.uint16), n * batch)
    m.setInput(x, batch)
    m.run(batch)
    took = []
    for pin in (True, False):
        buf = torch.zeros(n * batch, dtype=torch.int16, pin_memory=pin)
        best = 1e9
        for _ in range(6):
            t0 = time.perf_counter()
            assert ia.lib().ivh_read_output_f16(m._h, 0, buf.data_ptr(), batch) == 0
            best = min(best, time.perf_counter() - t0)
        assert np.array_equal(buf.numpy().view(np.uint16), x)
        took.append(best)
    dev = torch.zeros(n * batch, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    if ia.lib().ivh_read_output_f16(m._h, 0, dev.data_ptr(), batch) == 0:  # the runtime's copy takes it
        assert np.array_equal(dev.cpu().numpy().view(np.uint16), x)
    print(f"16 MB: pinned {took[0] * 1e6:.0f} us, pageable {took[1] * 1e6:.0f} us")
    m.close()
    assert took[0] < took[1]
