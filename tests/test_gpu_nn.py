"""Correction-network kernels (tsu_nn_* in include/tsuner.h) against the CPU
network oracle (oracle/nn_oracle.py), on BF16-rounded operands.

Tolerances: a BF16 output may differ from the FP64-accumulated oracle by one
BF16 rounding step (relative 2^-7) because the kernels accumulate in FP32;
FP32 outputs (the last layer, weight gradients) within 1e-5 of the largest
reference magnitude."""
import ctypes as C

import numpy as np
import pytest

import nn_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev_bf16(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(torch.bfloat16).cuda()


def dev_f32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.float().cpu().numpy()


_KEEP = []


def P(t):
    """Device address of t; t is kept alive until the test ends, so that
    temporaries passed inline are not recycled by the caching allocator while
    the enqueued kernels still use them."""
    _KEEP.append(t)
    return C.c_void_p(t.data_ptr())


@pytest.fixture(autouse=True)
def _release():
    yield
    torch.cuda.synchronize()
    _KEEP.clear()


def lib():
    from tsuner_amd import _lib
    return _lib.lib()


def ok(rc):
    from tsuner_amd import _lib
    _lib.check(rc, "call")


def assert_bf16_close(got, ref):
    err = np.abs(got - ref)
    tol = 2.0 ** -7 * np.abs(ref) + 1e-6 * max(1e-30, np.abs(ref).max())
    bad = err > tol
    assert not bad.any(), "max err %g at %s (ref %g got %g)" % (
        err.max(), np.argwhere(bad)[0], ref[tuple(np.argwhere(bad)[0])], got[tuple(np.argwhere(bad)[0])])


SHAPE = (2, 5, 70)     # n, h, w: two 64-pixel segments per row, one partial


def rand_bf16(rng, shape, scale=1.0):
    return O.bf16(rng.normal(0, scale, size=shape).astype(np.float32))


W64 = 16   # TSU_NN_W64


@pytest.mark.parametrize("width", [32, 64])
def test_mfma_conv_forward_kinds(width):
    rng = np.random.default_rng(1)
    n, h, w = SHAPE
    s = C.c_void_p(0)
    f = W64 if width == 64 else 0
    for kind, k, m, mreal in [(0, 8, width, width), (1, width, width, width), (2, width, 16, 4)]:
        x = rand_bf16(rng, (n, h, w, k))
        wt = rand_bf16(rng, (9, m, k), 0.2)
        if mreal < m:
            wt[:, mreal:, :] = 0
        b = rng.normal(0, 0.1, size=m).astype(np.float32)
        ref = O.conv(x, wt[:, :mreal, :], b[:mreal])
        if kind == 2:
            out = torch.zeros(n * h * w * 4, dtype=torch.float32, device="cuda")
        else:
            out = torch.zeros(n * h * w * m, dtype=torch.bfloat16, device="cuda")
        ok(lib().tsu_nn_conv(kind | f, P(dev_bf16(x)), P(dev_bf16(wt)), P(dev_f32(b)), None, P(out), n, h, w, s))
        got = host(out).reshape(n, h, w, -1)
        if kind == 2:
            np.testing.assert_allclose(got, ref, rtol=0, atol=1e-5 * np.abs(ref).max())
        else:
            assert_bf16_close(got, O.bf16(np.maximum(ref, 0).astype(np.float32)))


@pytest.mark.parametrize("width", [32, 64])
def test_mfma_conv_data_gradients_with_relu_mask(width):
    rng = np.random.default_rng(2)
    n, h, w = SHAPE
    s = C.c_void_p(0)
    f, W = (W64 if width == 64 else 0), width
    # through the output layer: dy has 8 channels (4 used), weights [9][16][W]
    w4 = rand_bf16(rng, (9, 16, W), 0.2)
    w4[:, 4:, :] = 0
    dy = np.zeros((n, h, w, 8), np.float32)
    dy[..., :4] = rand_bf16(rng, (n, h, w, 4))
    act = np.maximum(rand_bf16(rng, (n, h, w, W)), 0)
    wb = torch.zeros(9 * 16 * W, dtype=torch.bfloat16, device="cuda")
    wtr = torch.zeros(9 * W * 8, dtype=torch.bfloat16, device="cuda")
    ok(lib().tsu_nn_pack(P(dev_f32(w4)), P(wb), P(wtr), 16, W, 8, s))
    np.testing.assert_array_equal(host(wb).reshape(9, 16, W), w4)
    np.testing.assert_array_equal(host(wtr).reshape(9, W, 8), np.transpose(w4[:, :8, :], (0, 2, 1)))
    out = torch.zeros(n * h * w * W, dtype=torch.bfloat16, device="cuda")
    ok(lib().tsu_nn_conv(3 | f, P(dev_bf16(dy)), P(wtr), None, P(dev_bf16(act)), P(out), n, h, w, s))
    ref = O.conv_input_grad(dy[..., :4], w4[:, :4, :]) * (act > 0)
    assert_bf16_close(host(out).reshape(n, h, w, W), O.bf16(ref.astype(np.float32)))
    # middle layer
    w2 = rand_bf16(rng, (9, W, W), 0.2)
    d = rand_bf16(rng, (n, h, w, W))
    wt2 = torch.zeros(9 * W * W, dtype=torch.bfloat16, device="cuda")
    ok(lib().tsu_nn_pack(P(dev_f32(w2)), P(torch.zeros_like(wt2)), P(wt2), W, W, W, s))
    ok(lib().tsu_nn_conv(4 | f, P(dev_bf16(d)), P(wt2), None, P(dev_bf16(act)), P(out), n, h, w, s))
    ref = O.conv_input_grad(d, w2) * (act > 0)
    assert_bf16_close(host(out).reshape(n, h, w, W), O.bf16(ref.astype(np.float32)))


@pytest.mark.parametrize("width", [32, 64])
def test_mfma_weight_gradients(width):
    rng = np.random.default_rng(3)
    n, h, w = SHAPE
    s = C.c_void_p(0)
    f, W = (W64 if width == 64 else 0), width
    for kind, kx, my, mrows in [(5 | f, 8, W, W), (6 | f, W, W, W), (7 | f, W, 8, 16)]:
        x = rand_bf16(rng, (n, h, w, kx))
        dy = rand_bf16(rng, (n, h, w, my))
        dw = torch.full((9 * mrows * kx,), 7.0, dtype=torch.float32, device="cuda")
        db = torch.zeros(my, dtype=torch.float32, device="cuda")
        nws = lib().tsu_nn_wgrad_workspace(kind)
        ws = torch.zeros(nws, dtype=torch.float32, device="cuda")
        ok(lib().tsu_nn_wgrad(kind, P(dev_bf16(x)), P(dev_bf16(dy)), P(dw), P(db), mrows, n, h, w, P(ws), nws, s))
        rdw, rdb = O.conv_weight_grad(x, dy)
        got = host(dw).reshape(9, mrows, kx)
        np.testing.assert_allclose(got[:, :my, :], rdw, rtol=0, atol=1e-5 * np.abs(rdw).max())
        assert np.all(got[:, my:, :] == 7.0)      # rows beyond the gradient are left alone
        np.testing.assert_allclose(host(db), rdb, rtol=0, atol=1e-5 * np.abs(rdb).max())


@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 4, 64), (1, 9, 65), (3, 8, 63), (2, 26, 129), None])
def test_conv_strips_and_stretches(shape, width):
    """The convolutions walk 64-column strips in passes of 4 or 8 rows through
    an LDS ring: images smaller than a pass, a column past a strip, rows past
    a pass, several turns of the ring, and (None) more passes than
    workgroups, so that stretches start and end inside strips.  Tolerances as
    for the single kinds (one BF16 rounding step; FP32 output 1e-5)."""
    rng = np.random.default_rng(15)
    s = C.c_void_p(0)
    f, W = (W64 if width == 64 else 0), width
    for kind, k, m in [(0, 8, W), (1, W, W), (2, W, 4), (3, 8, W), (4, W, W)]:
        n, h, w = shape or ((58 if k == 8 else 15), 45, 150)
        x = rand_bf16(rng, (n, h, w, k))
        rows = 16 if kind == 2 else m
        wt = rand_bf16(rng, (9, rows, k), 0.2)
        wt[:, m:] = 0
        b = rng.normal(0, 0.1, size=64).astype(np.float32)
        act = np.maximum(rand_bf16(rng, (n, h, w, m)), 0)
        out = torch.full((n * h * w * m,), 9.0, dtype=torch.float32 if kind == 2 else torch.bfloat16, device="cuda")
        ok(lib().tsu_nn_conv(kind | f, P(dev_bf16(x)), P(dev_bf16(wt)), P(dev_f32(b)), P(dev_bf16(act)), P(out), n, h,
                             w, s))
        got = host(out).reshape(n, h, w, m)
        if kind >= 3:      # the kernel's weights are the per-tap transposes: out[p] = sum_t wt[t] in[p - off(t)]
            ref = O.conv_input_grad(x, np.transpose(wt, (0, 2, 1))) * (act > 0)
        else:
            ref = O.conv(x, wt[:, :m], b[:m])
        if kind == 2:
            np.testing.assert_allclose(got, ref, rtol=0, atol=1e-5 * np.abs(ref).max())
        else:
            assert_bf16_close(got, O.bf16((np.maximum(ref, 0) if kind < 2 else ref).astype(np.float32)))


@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 4, 64), (1, 9, 65), (3, 8, 63), (2, 17, 130), (15, 45, 150)])
def test_weight_gradient_strips_and_stretches(shape, width):
    """The weight-gradient kernels walk 64-column strips in passes of 4 or 8
    rows, cut into at most 256 stretches: images smaller than a pass, a
    column past a strip, rows past a pass, and (the last shape) more passes
    than stretches for every kind, so that stretches start and end inside
    strips.  Tolerance: FP32 accumulation over P pixels in chains of at most
    P / 32 + 256 additions errs by about 6e-8 sqrt(P / 32 + 256) of a partial
    sum that itself is of the size of the largest entry, below 1e-5 here."""
    rng = np.random.default_rng(13)
    n, h, w = shape
    s = C.c_void_p(0)
    f, W = (W64 if width == 64 else 0), width
    for kind, kx, my, mrows in [(5 | f, 8, W, W), (6 | f, W, W, W), (7 | f, W, 8, 16)]:
        x = rand_bf16(rng, (n, h, w, kx))
        dy = rand_bf16(rng, (n, h, w, my))
        dw = torch.full((9 * mrows * kx,), 7.0, dtype=torch.float32, device="cuda")
        db = torch.zeros(my, dtype=torch.float32, device="cuda")
        nws = lib().tsu_nn_wgrad_workspace(kind)
        ws = torch.full((nws,), float("nan"), dtype=torch.float32, device="cuda")
        ok(lib().tsu_nn_wgrad(kind, P(dev_bf16(x)), P(dev_bf16(dy)), P(dw), P(db), mrows, n, h, w, P(ws), nws, s))
        rdw, rdb = O.conv_weight_grad(x, dy)
        got = host(dw).reshape(9, mrows, kx)
        np.testing.assert_allclose(got[:, :my, :], rdw, rtol=0, atol=1e-5 * np.abs(rdw).max())
        assert np.all(got[:, my:, :] == 7.0)
        np.testing.assert_allclose(host(db), rdb, rtol=0, atol=1e-5 * np.abs(rdb).max())


@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 5, 9), (1, 9, 65), (1, 8, 64), (2, 11, 130)])
def test_weight_gradients_of_values_that_are_not_finite(shape, width):
    """dW[t] = sum_p dy[p] x[p + t] with zeros for x around the image and p
    over the image alone, for an infinity or a NaN of x, of dy and of both on
    the image's border and inside: the same entries are infinite, of the same
    sign, and NaN as in the oracle's sum, and the others are right (tolerance
    as above)."""
    rng = np.random.default_rng(22)
    n, h, w = shape
    s = C.c_void_p(0)
    f, W = (W64 if width == 64 else 0), width
    spots = sorted({(r, c) for r in (0, h // 2, h - 1) for c in (0, w // 2, w - 1)})
    for kind, kx, my in [(5 | f, 8, W), (6 | f, W, W), (7 | f, W, 8)]:
        nws = lib().tsu_nn_wgrad_workspace(kind)
        ws = torch.empty(nws, dtype=torch.float32, device="cuda")
        for at in spots:
            for which in (1, 2, 3):
                x = rand_bf16(rng, (n, h, w, kx))
                dy = rand_bf16(rng, (n, h, w, my))
                if which & 1:
                    x[n - 1, at[0], at[1], 3] = [np.inf, -np.inf, np.nan][rng.integers(3)]
                if which & 2:
                    r, c = (at if rng.integers(2) else spots[rng.integers(len(spots))])
                    dy[n - 1, r, c, 1] = [np.inf, -np.inf, np.nan][rng.integers(3)]
                dw = torch.zeros(9 * my * kx, dtype=torch.float32, device="cuda")
                db = torch.zeros(my, dtype=torch.float32, device="cuda")
                ok(lib().tsu_nn_wgrad(kind, P(dev_bf16(x)), P(dev_bf16(dy)), P(dw), P(db), my, n, h, w, P(ws), nws, s))
                with np.errstate(invalid="ignore"):
                    rdw, rdb = O.conv_weight_grad(x, dy)
                for got, ref in ((host(dw).reshape(9, my, kx), rdw), (host(db), rdb)):
                    fin = np.isfinite(ref)
                    np.testing.assert_array_equal(got[~fin], ref[~fin].astype(np.float32))
                    if fin.any():
                        np.testing.assert_allclose(got[fin], ref[fin], rtol=0, atol=1e-5 * np.abs(ref[fin]).max())
        _KEEP.clear()


def test_weight_gradients_take_operands_of_any_alignment():
    """x and dy one element past a 16-byte boundary: the same sums, bit for
    bit, as from aligned copies."""
    rng = np.random.default_rng(14)
    n, h, w = 2, 9, 70
    s = C.c_void_p(0)
    for kind, kx, my in [(5, 8, 32), (6 | W64, 64, 64), (7, 32, 8)]:
        nws = lib().tsu_nn_wgrad_workspace(kind)
        ws = torch.zeros(nws, dtype=torch.float32, device="cuda")
        x = dev_bf16(rand_bf16(rng, n * h * w * kx))
        dy = dev_bf16(rand_bf16(rng, n * h * w * my))
        got = []
        for shift in (0, 1):
            tx, ty = (torch.zeros(t.numel() + shift, dtype=t.dtype, device="cuda") for t in (x, dy))
            tx[shift:].copy_(x)
            ty[shift:].copy_(dy)
            dw = torch.zeros(9 * my * kx, dtype=torch.float32, device="cuda")
            db = torch.zeros(my, dtype=torch.float32, device="cuda")
            ok(lib().tsu_nn_wgrad(kind, P(tx[shift:]), P(ty[shift:]), P(dw), P(db), my, n, h, w, P(ws), nws, s))
            got.append((host(dw), host(db)))
        assert np.abs(got[0][0]).max() > 0
        np.testing.assert_array_equal(got[1][0], got[0][0])
        np.testing.assert_array_equal(got[1][1], got[0][1])


def test_wide_conv_workgroups_loop_over_tiles():
    """The 64-channel kernels keep one workgroup per CU and loop over 8 x 64
    pixel tiles (prefetching the next one): an image set with more than
    twice as many tiles as CUs, ragged in both directions, against the
    oracle, forward and data gradient."""
    rng = np.random.default_rng(9)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    h, w = 45, 150                      # 6 x 3 tiles per image, partial ones at both edges
    n = (2 * cus) // 18 + 1
    s = C.c_void_p(0)
    x = rand_bf16(rng, (n, h, w, 64))
    wt = rand_bf16(rng, (9, 64, 64), 0.1)
    b = rng.normal(0, 0.1, size=64).astype(np.float32)
    out = torch.zeros(n * h * w * 64, dtype=torch.bfloat16, device="cuda")
    ok(lib().tsu_nn_conv(1 | W64, P(dev_bf16(x)), P(dev_bf16(wt)), P(dev_f32(b)), None, P(out), n, h, w, s))
    assert_bf16_close(host(out).reshape(n, h, w, 64), O.bf16(np.maximum(O.conv(x, wt, b), 0).astype(np.float32)))
    act = np.maximum(rand_bf16(rng, (n, h, w, 64)), 0)
    wtr = torch.zeros(9 * 64 * 64, dtype=torch.bfloat16, device="cuda")
    ok(lib().tsu_nn_pack(P(dev_f32(wt)), P(torch.zeros_like(wtr)), P(wtr), 64, 64, 64, s))
    ok(lib().tsu_nn_conv(4 | W64, P(dev_bf16(x)), P(wtr), None, P(dev_bf16(act)), P(out), n, h, w, s))
    ref = O.conv_input_grad(x, wt) * (act > 0)
    assert_bf16_close(host(out).reshape(n, h, w, 64), O.bf16(ref.astype(np.float32)))


@pytest.mark.parametrize("width", [32, 64])
def test_output_layer_takes_four_biases(width):
    """The output layer's bias is four values (its weights are 16 rows); what
    lies behind them in memory is not the layer's and changes nothing.
    Tolerance as for the single kinds (FP32 output 1e-5)."""
    rng = np.random.default_rng(21)
    n, h, w = 2, 6, 70
    x = rand_bf16(rng, (n, h, w, width))
    wt = rand_bf16(rng, (9, 16, width), 0.2)
    wt[:, 4:] = 0
    b = rng.normal(0, 0.1, size=4).astype(np.float32)
    room = dev_f32(np.concatenate([b, np.full(12, np.nan, np.float32)]))
    out = torch.zeros(n * h * w * 4, dtype=torch.float32, device="cuda")
    ok(lib().tsu_nn_conv(2 | (W64 if width == 64 else 0), P(dev_bf16(x)), P(dev_bf16(wt)), P(room[:4]), None, P(out), n,
                         h, w, C.c_void_p(0)))
    ref = O.conv(x, wt[:, :4], b)
    np.testing.assert_allclose(host(out).reshape(ref.shape), ref, rtol=0, atol=1e-5 * np.abs(ref).max())


def test_mse_and_adam_kernels():
    rng = np.random.default_rng(4)
    npix = 1000
    out = rng.normal(size=(npix, 4)).astype(np.float32)
    tgt = rng.normal(size=(npix, 4)).astype(np.float32)
    dy = torch.zeros(npix * 8, dtype=torch.bfloat16, device="cuda")
    lp = torch.zeros(64, dtype=torch.float64, device="cuda")
    ok(lib().tsu_nn_mse(P(dev_f32(out)), P(dev_f32(tgt)), P(dy), P(lp), 64, npix, C.c_float(0.5), C.c_void_p(0)))
    g = host(dy).reshape(npix, 8)
    np.testing.assert_array_equal(g[:, :4], O.bf16((0.5 * (out - tgt)).astype(np.float32)))
    assert np.all(g[:, 4:] == 0)
    d = (out - tgt).astype(np.float64)
    np.testing.assert_allclose(lp.cpu().numpy().sum(), (d * d).sum(), rtol=1e-12)
    # Adam: one step from m = v = 0 moves every parameter by lr_t * sign-ish
    p = rng.normal(size=300).astype(np.float32)
    gr = rng.normal(size=300).astype(np.float32)
    tp, tg = dev_f32(p), dev_f32(gr)
    tm, tv = torch.zeros_like(tp), torch.zeros_like(tp)
    ok(lib().tsu_nn_adam(P(tp), P(tg), P(tm), P(tv), 300, C.c_float(1e-2), C.c_float(0.9), C.c_float(0.999),
                         C.c_float(1e-8), C.c_void_p(0)))
    # the kernel's FP32 constants: (1 - 0.9f) and (1 - 0.999f) are not 0.1 and 0.001
    one, b1, b2 = np.float32(1), np.float32(0.9), np.float32(0.999)
    m = (one - b1) * gr
    v = (one - b2) * gr * gr
    np.testing.assert_allclose(host(tm), m, rtol=1e-6)
    np.testing.assert_allclose(host(tv), v, rtol=1e-6)
    np.testing.assert_allclose(host(tp), p - np.float32(1e-2) * m / (np.sqrt(v) + np.float32(1e-8)), rtol=1e-5,
                               atol=1e-7)


@pytest.mark.parametrize("width,mids", [(32, 0), (32, 2), (64, 1), (64, 4)])
def test_adam_pack_equals_step_and_packs(width, mids):
    """One launch for the step and all layers' BF16 copies against the step
    and one packing per layer: the same values."""
    import math
    import torch
    from tsuner_amd import nn
    arch = nn.Arch(width, mids)
    rng = np.random.default_rng(width + mids)
    g, m, v = (rng.normal(size=arch.nparam).astype(np.float32) for _ in range(3))
    nets = [nn.Net(nn.init_params(3, arch), max_batch=1, h=8, w=8, arch=arch) for _ in range(2)]
    for net in nets:
        net.g.copy_(dev_f32(g))
        net.m.copy_(dev_f32(1e-3 * m))
        net.v.copy_(dev_f32(1e-6 * v * v))
    a, b = nets
    a.adam(1e-2)
    lr_t = 1e-2 * math.sqrt(1.0 - 0.999) / (1.0 - 0.9)
    ok(lib().tsu_nn_adam(P(b.p), P(b.g), P(b.m), P(b.v), arch.nparam, C.c_float(lr_t), C.c_float(0.9), C.c_float(0.999),
                         C.c_float(1e-8), C.c_void_p(0)))
    b.pack()
    for x, y in zip([a.p, a.m, a.v] + a.wb + a.wt[1:], [b.p, b.m, b.v] + b.wb + b.wt[1:]):
        assert torch.equal(x, y)
    assert not torch.equal(a.p, dev_f32(nn.init_params(3, arch)))
    s = C.c_void_p(0)
    assert lib().tsu_nn_adam_pack(P(a.p), P(a.g), P(a.m), P(a.v), C.c_float(0), C.c_float(0), C.c_float(0), C.c_float(1),
                                  48, 1, P(a.p), P(a.p), s) != 0


@pytest.mark.parametrize("width,mids", [(32, 2), (64, 1), (32, 4)])
def test_network_gradients_match_oracle(width, mids):
    """Full forward + backward on the GPU against the oracle's loss_and_grads
    (pinned by finite differences in test_nn_oracle.py), run with BF16
    rounding at the points where the GPU stores BF16 (hidden activations, the
    output gradient, the masked data gradients): norm-wise 1% per tensor, the
    rest being FP32 accumulation and the rare BF16 rounding flips it causes.
    Against the unrounded FP64 oracle the same gradients agree to 8%."""
    from tsuner_amd import nn
    arch = nn.Arch(width, mids)
    last = arch.nlayers - 1
    rng = np.random.default_rng(5)
    n, h, w = 2, 12, 20
    p = nn.init_params(7, arch)
    # give the output layer full-size weights so every layer carries gradient
    wo, bo = arch.offs[last]
    p[wo:wo + 9 * 16 * width] *= 10.0
    for li, (m, k) in enumerate(arch.layers):
        p[arch.offs[li][1]:arch.offs[li][1] + m] = rng.normal(0, 0.05, m)
    p[bo + 4:bo + 16] = 0
    p = O.bf16(p)
    net = nn.Net(p, max_batch=n, h=h, w=w, arch=arch)
    x = rand_bf16(rng, (n, h, w, 8))
    tgt = rng.normal(0, 1, size=(n, h, w, 4)).astype(np.float32)
    tx, tt = dev_bf16(x), dev_f32(tgt)
    net.forward(tx, n)
    net.backward(tx, tt, n)
    gpu_loss = net.loss(n)
    g = net.g.cpu().numpy()
    params = []
    for li, (m, k) in enumerate(arch.layers):
        wo, bo = arch.offs[li]
        W = p[wo:wo + 9 * m * k].reshape(9, m, k).astype(np.float64)
        b = p[bo:bo + m].astype(np.float64)
        if li == last:
            W, b = W[:, :4, :], b[:4]
        params.append((W, b))
    loss, grads = O.loss_and_grads(x.astype(np.float64), tgt.astype(np.float64), params, rnd=O.bf16_64)
    loss64, grads64 = O.loss_and_grads(x.astype(np.float64), tgt.astype(np.float64), params)
    assert abs(gpu_loss - loss) <= 1e-3 * loss
    for li, (m, k) in enumerate(arch.layers):
        wo, bo = arch.offs[li]
        gw = g[wo:wo + 9 * m * k].reshape(9, m, k)
        gb = g[bo:bo + m]
        if li == last:
            assert np.all(gw[:, 4:, :] == 0) and np.all(gb[4:] == 0)
            gw, gb = gw[:, :4, :], gb[:4]
        for (rw, rb), tol in ((grads[li], 0.01), (grads64[li], 0.08)):
            assert np.linalg.norm(gw - rw) <= tol * np.linalg.norm(rw), (li, tol)
            assert np.linalg.norm(gb - rb) <= tol * np.linalg.norm(rb), (li, tol)


def test_training_reduces_loss():
    """Adam on the GPU fits a target produced by a fixed random network of
    the same shape (realisable): the loss falls by 10x."""
    from tsuner_amd import nn
    rng = np.random.default_rng(6)
    n, h, w = 4, 16, 24
    teacher = nn.Net(nn.init_params(11), max_batch=n, h=h, w=w)
    x = dev_bf16(rand_bf16(rng, (n, h, w, 8)))
    tgt = teacher.forward(x, n).clone()
    student = nn.Net(nn.init_params(12), max_batch=n, h=h, w=w)
    student.forward(x, n)
    student.backward(x, tgt, n)
    first = student.loss(n)
    for _ in range(300):
        student.train_step(x, tgt, n, lr=3e-3)
    student.forward(x, n)
    student.backward(x, tgt, n)
    assert student.loss(n) < 0.1 * first, (first, student.loss(n))
