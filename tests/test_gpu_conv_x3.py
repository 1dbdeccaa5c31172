"""The convolutions on the bf16 matrix cores (F32 operands as exact sums of
three bf16 values, conv_x3.hip), reached through levo_hip_snake_conv1d_split,
levo_hip_snake_conv_transpose1d_split and levo_hip_vae_decode where the launch
is large enough and the workspace holds the split weights.

Bars: max |y - exact| / max(|exact|, 1) <= 1e-5 against the convolution of the
oracle's SnakeBeta output in float64, the bar of the F32 launches, and in the
2-norm no further from it than the F32 launch of the same data (the split
operands are exact, the products left out are below 2^-24 of a product, and the
sums round once per 16 terms where the F32 MFMA rounds once per 4). The route is
checked too: another order of the sums gives other bits than the F32 launch,
whose grid is full where a test says that the epilogue is the direct one.
Shapes: partial row tiles (129, 200, 257 output channels) and channel groups,
column tiles of 128 (127 for the transposed form) with remainders, the widest
halo (dilation 10) and the first beyond it (11, which keeps the F32 launch),
strides, F16 parameters, arguments beyond the reduced sine, y over the residual,
each with partial sums (the queried workspace) and in one split (`direct`);
whole decodes of windows that take every form; special, tiny and huge values.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f32_err, from_dev, to_dev
from test_gpu_snake_conv_split import _case, _f64_rows, _f64_transpose_rows, _run, _run_t, _t_case
from test_gpu_vae_decoder import device_weights
from vae_chain import Weights, decode_f64, scaled_err

pytestmark = pytest.mark.gpu


def _direct_floats(c_in, rows, kw, cols):
    """Workspace for the split weights and less than two partial sums: one split, the direct epilogue."""
    pack = -(-rows // 32) * 32 * -(-c_in // 32) * 32 * kw * 3 // 2
    return pack + pack // 64 + 8 * (c_in + rows) + 64 + rows * cols


def _compare(got, plain, exact, rows):
    assert f32_err(got[rows], exact) <= 1e-5
    assert np.linalg.norm(got[rows] - exact) <= np.linalg.norm(plain[rows] - exact)
    assert not np.array_equal(got.view(np.uint32), plain.view(np.uint32))


@pytest.mark.parametrize("c_in,c_out,t,kw,dil,residual", [
    (256, 256, 12001, 7, 1, False), (512, 512, 9001, 7, 3, True), (130, 200, 9999, 7, 10, False),
    (1021, 257, 5003, 7, 1, False), (250, 256, 40003, 3, 9, True), (512, 512, 15121, 1, 1, True),
    (1000, 129, 20001, 1, 1, False)])
def test_conv(hip, dev, oracle, c_in, c_out, t, kw, dil, residual):
    pad = dil * (kw - 1) // 2
    x, w, b, a, bl, r = _case(oracle, c_in, c_out, t, kw, c_in + t, residual)
    got = _run(hip, dev, x, w, b, pad, dil, a, bl, r)
    plain = _run(hip, dev, x, w, b, pad, dil, a, bl, r, ws_floats=None)
    rows = np.arange(0, c_out, 16)
    _compare(got, plain, _f64_rows(oracle, x, w, b, pad, dil, a, bl, r, rows), rows)
    again = _run(hip, dev, x, w, b, pad, dil, a, bl, r)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))


@pytest.mark.parametrize("c_in,c_out,t_in,stride,pad", [(1024, 512, 2521, 6, 3), (512, 256, 3001, 4, 2),
                                                        (128, 128, 40003, 2, 1), (300, 200, 5001, 3, 2),
                                                        (256, 130, 16257, 5, 0)])
def test_transpose(hip, dev, oracle, c_in, c_out, t_in, stride, pad):
    x, w, b, a, bl = _t_case(oracle, c_in, c_out, t_in, stride, c_in + t_in)
    got = _run_t(hip, dev, x, w, b, stride, pad, a, bl)
    plain = _run_t(hip, dev, x, w, b, stride, pad, a, bl, split=False)
    rows = np.arange(0, c_out, 16)
    _compare(got, plain, _f64_transpose_rows(oracle, x, w, b, stride, pad, a, bl, rows), rows)


def test_falls_back(hip, dev, oracle):
    """Dilation 11 (a halo of 66 columns; room for one partial sum, so no split
    either) and a workspace short of the split weights keep the F32 launch, bit
    for bit."""
    c, t = 256, 33000
    x, w, b, a, bl, _ = _case(oracle, c, c, t, 7, 5)
    for dil, n in ((11, c * t), (3, c * c * 7)):
        got = _run(hip, dev, x, w, b, 3 * dil, dil, a, bl, ws_floats=n)
        plain = _run(hip, dev, x, w, b, 3 * dil, dil, a, bl, ws_floats=None)
        assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))


@pytest.mark.parametrize("c_in,kw", [(1, 3), (2, 1)])
def test_sums_of_few_terms_stay_in_f32(hip, dev, c_in, kw):
    """Below four terms the F32 launch is the closer one: its bits."""
    import torch
    c_out = 512
    t = 420_000_000 // (c_out * c_in * kw)
    g = torch.Generator(device=dev).manual_seed(4)
    x, w = torch.randn(c_in, t, device=dev, generator=g), torch.randn(c_out, c_in, kw, device=dev, generator=g)
    got, plain = torch.empty(c_out, t, device=dev), torch.empty(c_out, t, device=dev)
    ws = torch.empty(4 * c_out * kw * 64, device=dev)  # the split weights and no partial sum
    hip.snake_conv1d_split(x, c_in, t, w, c_out, kw, workspace=ws, workspace_floats=ws.numel(), padding=kw // 2, y=got)
    hip.snake_conv1d(x, c_in, t, w, c_out, kw, padding=kw // 2, y=plain)
    assert torch.equal(got, plain)


@pytest.mark.parametrize("t,direct", [(12345, False), (16741, True)])
def test_f16_params_large_arguments_in_place_residual(hip, dev, oracle, t, direct):
    """|alpha x| beyond the reduced sine's 8192 in some channels; y written over
    the residual."""
    c = 256
    x, w, b, a, bl, r = _case(oracle, c, c, t, 7, 9, True)
    x[::5, ::7] *= np.float32(3e4)
    a16, b16 = oracle.f32_to_f16(a), oracle.f32_to_f16(bl)
    a32, b32 = oracle.f16_to_f32(a16), oracle.f16_to_f32(b16)
    got = _run(hip, dev, x, w, b, 9, 3, a16, b16, r, param_type=1, in_place=True,
               ws_floats=_direct_floats(c, c, 7, t) if direct else -1)
    plain = _run(hip, dev, x, w, b, 9, 3, a16, b16, r, param_type=1, ws_floats=None)
    rows = np.arange(0, c, 16)
    exact = _f64_rows(oracle, x, w, b, 9, 3, a32, b32, r, rows)
    # the signal is 1e4 times larger than a unit one: errors relative to its largest value
    assert np.max(np.abs(got[rows] - exact)) <= 1e-5 * np.max(np.abs(exact))
    assert np.linalg.norm(got[rows] - exact) <= np.linalg.norm(plain[rows] - exact)


@pytest.mark.parametrize("t,direct", [(12001, False), (16641, True)])
def test_strides(hip, dev, oracle, t, direct):
    """x, residual and y rows further apart than their samples, none aligned."""
    import torch
    c, kw = 256, 7
    x, w, b, a, bl, r = _case(oracle, c, c, t, kw, 11, True)
    xd = torch.full((c, t + 5), float("nan"), device=dev)
    rd = torch.full((c, t + 3), float("nan"), device=dev)
    yd = torch.full((c, t + 9), 7.0, device=dev)
    xd[:, :t], rd[:, :t] = to_dev(x, dev), to_dev(r, dev)
    n = _direct_floats(c, c, kw, t) if direct else hip.snake_conv1d_split_workspace_floats(c, t)
    ws = torch.full((n,), float("nan"), device=dev)
    hip.snake_conv1d_split(xd, c, t, to_dev(w, dev), c, kw, workspace=ws, workspace_floats=n, x_stride=t + 5,
                           alpha_log=to_dev(a, dev), beta_log=to_dev(bl, dev), bias=to_dev(b, dev), padding=3,
                           residual=rd, residual_stride=t + 3, y=yd, y_stride=t + 9)
    torch.cuda.synchronize()
    got = from_dev(yd)
    assert np.array_equal(got[:, :t], _run(hip, dev, x, w, b, 3, 1, a, bl, r, ws_floats=n))
    assert not np.array_equal(got[:, :t], _run(hip, dev, x, w, b, 3, 1, a, bl, r, ws_floats=None))
    assert np.all(got[:, t:] == 7.0)


@pytest.mark.parametrize("kw,where,direct,snake", [
    (7, "x", False, False), (1, "x", False, False), (7, "w", False, False), (2, "x", False, False), (2, "w", False, False),
    (7, "x", True, False), (7, "w", True, True), (2, "x", True, True), (2, "w", True, False), (7, "x", True, True),
    (7, "x", False, True), (1, "w", True, True), (7, "w not finite", True, True), (2, "w not finite", False, False),
    (7, "w not finite", False, False), (1, "w not finite", True, False)])
def test_values_that_cannot_be_split(hip, dev, oracle, kw, where, direct, snake):
    """Infinities, NaN and a finite value that rounds to a bf16 infinity, in the
    input and in the weights, with SnakeBeta (which makes NaN of an infinity) and
    without: the same infinities and NaN as the F32 launch, the other outputs
    within the F32 bar."""
    c, t = (256, 20000) if kw != 2 else (512, 4300)
    big = (np.inf, -np.inf, np.nan, np.float32(3.4e38))[:3 if where == "w not finite" else 4]
    if kw == 2:
        x, w, b, a, bl = _t_case(oracle, c, 256, t, 4, 21)
    else:
        x, w, b, a, bl, _ = _case(oracle, c, c, t, kw, 21)
    if not snake:
        a = bl = None
    n = _direct_floats(c, c if kw != 2 else 1024, kw, t + 1) if direct else -1
    for i, v in enumerate(big):
        if where == "x":
            x[3 + 17 * i, 100 + 700 * i] = v
        elif kw == 2:
            w[3 + 17 * i, 5 + 40 * i, i] = v
        else:
            w[5 + 40 * i, 3 + 17 * i, i % kw] = v
    if kw == 2:
        got = _run_t(hip, dev, x, w, b, 4, 2, a, bl, ws_floats=n)
        plain = _run_t(hip, dev, x, w, b, 4, 2, a, bl, split=False)
    else:
        got, plain = (_run(hip, dev, x, w, b, kw // 2, 1, a, bl, ws_floats=m) for m in (n, None))
    # the bf16 route: other bits where all is finite (3.4e38 in the weights has every tile summed in F32)
    assert where == "w" or not np.array_equal(got[:, 4000:].view(np.uint32), plain[:, 4000:].view(np.uint32))
    _same_or_close(got, plain)


def _same_or_close(got, plain):
    """The infinities and NaN of the F32 launch, its other values to F32 rounding at their size."""
    assert not np.all(np.isfinite(plain))
    assert np.array_equal(np.isnan(got), np.isnan(plain))
    inf = np.isinf(plain)
    assert np.array_equal(inf, np.isinf(got)) and np.array_equal(np.sign(got[inf]), np.sign(plain[inf]))
    ok = np.isfinite(plain)
    # a sum with a term of 3e38 is as large: relative to the value there
    assert np.max(np.abs(got[ok].astype(np.float64) - plain[ok]) / np.maximum(np.abs(plain[ok]), 1.0)) <= 2e-5


# 2^64 (1 - 2^-10) squared is finite, the product of its bf16 roundings is not
EDGE = np.float32(2.0 ** 64 * (1 - 2.0 ** -10))
OVERFLOWS = [(1e30, -1e14), (1e30, 1e14), (1.003e25, 1.003e20), (-1e25, 1e20), (1.005e25, 1.001e20), (EDGE, EDGE)]


@pytest.mark.parametrize("direct", [True, False])
@pytest.mark.parametrize("kw", [7, 1, 3, 2])
def test_products_that_overflow(hip, dev, oracle, kw, direct):
    """Finite operands whose products pass the largest F32 (by far, where the
    parts of the split operands overflow with either sign, and by so little that
    only the product of their first parts does): the infinities, NaN and finite
    values of the F32 launch, in one split and in several."""
    c, c_out, t, stride = (256, 256, 20000, 1) if kw != 2 else (512, 256, 4300, 4)
    if kw == 2:
        x, w, b, _, _ = _t_case(oracle, c, c_out, t, stride, 31)
    else:
        x, w, b, _, _, _ = _case(oracle, c, c_out, t, kw, 31)
    for i, (xv, wv) in enumerate(OVERFLOWS):
        x[3 + 17 * i, 100 + 400 * i] = xv
        if kw == 2:
            w[3 + 17 * i, 5 + 40 * i, i] = wv
        else:
            w[5 + 40 * i, 3 + 17 * i, i % kw] = wv
    n = _direct_floats(c, c_out * stride, kw, t + 1) if direct else -1
    if kw == 2:
        got, plain = _run_t(hip, dev, x, w, b, 4, 2, ws_floats=n), _run_t(hip, dev, x, w, b, 4, 2, split=False)
    else:
        got, plain = (_run(hip, dev, x, w, b, kw // 2, 1, ws_floats=m) for m in (n, None))
    assert not np.array_equal(got[:, 3000:].view(np.uint32), plain[:, 3000:].view(np.uint32))  # the bf16 route
    _same_or_close(got, plain)


def _decode(hip, dev, dw, latent, frames, stage5):
    import torch
    nbytes = hip.vae_decode_workspace_bytes(frames)
    ws = torch.full((nbytes // 4,), float("nan"), device=dev)
    audio = torch.empty(2, 1920 * frames, device=dev)
    out = torch.empty(128, 1920 * frames, device=dev) if stage5 else None
    hip.vae_decode(dw, to_dev(latent, dev), frames, audio, ws, nbytes, stage_outputs=[None] * 4 + [out] if stage5 else None)
    torch.cuda.synchronize()
    return from_dev(out if stage5 else audio)


def _f64_decode(w, latent, dev):
    """vae_chain's decode_f64 with torch on the GPU: one product per tap."""
    import torch
    put = lambda a: to_dev(a, dev).double()

    def snake(x, ab):
        return x + torch.sin(torch.exp(put(ab[0]))[:, None] * x) ** 2 / (torch.exp(put(ab[1])) + 1e-9)[:, None]

    def conv(x, wt, bias, dil):
        k, t = wt.shape[2], x.shape[1]
        xp = torch.nn.functional.pad(x, (dil * (k - 1) // 2, dil * (k - 1) // 2))
        y = sum(put(wt[:, :, j]) @ xp[:, j * dil:j * dil + t].contiguous() for j in range(k))
        return y if bias is None else y + put(bias)[:, None]

    def upsample(x, wt, bias, stride):
        t = x.shape[1]
        full = x.new_zeros(wt.shape[1], t + 1, stride)
        for r in range(stride):
            full[:, :t, r] += put(wt[:, :, r].T) @ x
            full[:, 1:, r] += put(wt[:, :, r + stride].T) @ x
        pad = (stride + 1) // 2
        return full.reshape(wt.shape[1], -1)[:, pad:(t + 1) * stride - pad] + put(bias)[:, None]

    h = conv(put(latent), *w.input, 1)
    for stage, stride in zip(w.stages, (10, 6, 4, 4, 2)):
        h = upsample(snake(h, stage["act"]), *stage["up"], stride)
        for unit, dil in zip(stage["res"], (1, 3, 9)):
            h = h + conv(snake(conv(snake(h, unit["pre"]), *unit["conv0"], dil), unit["post"]), *unit["conv1"], 1)
    return conv(snake(h, w.out_act), w.out_w, None, 1)


@pytest.mark.parametrize("frames", [7, 17, 24, 64, 110, 252, 1000])
def test_decoder(hip, binding, dev, oracle, frames):
    """Windows of every route (test_decoder_takes_every_form) against float64:
    the decoder's bar at the signal's scale, and in the 2-norm 1.2e-6, which the
    F32 launches keep to."""
    import torch
    w = Weights(binding, 50 + frames)
    latent = oracle.gaussian(64 * frames, frames).reshape(64, frames)
    dw, keep = device_weights(hip, binding, dev, w)
    got = _decode(hip, dev, dw, latent, frames, False).astype(np.float64)
    exact = _f64_decode(w, latent, dev).cpu().numpy()
    if frames == 7:
        assert scaled_err(exact, decode_f64(w, latent)) <= 1e-12
    assert scaled_err(got, exact) <= 1e-5
    assert np.linalg.norm(got - exact) <= 1.2e-6 * np.linalg.norm(exact)


def test_decoder_takes_every_form(hip, binding, dev, oracle):
    """The launches of the windows above: k = 7 and k = 1 convolutions of stages 1
    to 3 and the upsamplers with partial sums and without, the units of stages 4
    and 5, both narrow outputs, the thin upsampler."""
    import re
    import torch
    from torch.profiler import ProfilerActivity, profile
    w = Weights(binding, 51)
    dw, keep = device_weights(hip, binding, dev, w)
    forms = {}
    for frames in (7, 24, 110, 252, 1000):
        latent = oracle.gaussian(64 * frames, frames).reshape(64, frames)
        _decode(hip, dev, dw, latent, frames, False)
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            _decode(hip, dev, dw, latent, frames, False)
        events = sorted((e for e in prof.events() if "levo_hip::" in e.name), key=lambda e: e.time_range.start)
        if not events:
            pytest.skip("no kernel events from the profiler")
        names = [re.sub(r"\(anonymous namespace\)::|levo_hip::|void |\(.*", "", e.name.replace("(anonymous namespace)::", ""))
                 for e in events]
        forms[frames] = {n + (" + combine" if i + 1 < len(names) and "combine" in names[i + 1] else "")
                         for i, n in enumerate(names)}
    k7, k1, up, unit = ("x3_conv_kernel<%s>" % a for a in ("7, true, false", "1, false, false", "2, true, false",
                                                           "7, true, true"))
    assert {"thin_transpose_kernel<8>", k7 + " + combine", up + " + combine", unit,
            "snake_conv_narrow_kernel<7, 2, 1>"} <= forms[7]
    assert {k7 + " + combine", up + " + combine"} <= forms[24]
    assert {k7, k7 + " + combine", k1, k1 + " + combine", up, up + " + combine"} <= forms[110]
    assert {k7, k1, up, unit, "snake_conv_narrow_kernel<7, 2, 4>"} <= forms[252]
    assert {k7, k1, up, unit} <= forms[1000] and not any("scatter" in n for n in forms[1000])


@pytest.mark.parametrize("frames", [24, 110])
def test_stage_with_large_inner_values(hip, binding, dev, oracle, frames):
    """Stage 3 with values between its convolutions whose sine arguments pass the
    reduced form's range: the SnakeBeta that the k = 7 convolution stores is
    evaluated anew there, in the combine (24 frames) and in the direct epilogue
    (110). Against the public F32 calls from the decode's own stage 2 output."""
    w = Weights(binding, 90)
    for unit in w.stages[2]["res"]:
        unit["conv0"][1][::9] = np.float32(3e4)
        unit["conv1"][0][:, ::9] *= np.float32(1e-4)
    latent = oracle.gaussian(64 * frames, 13).reshape(64, frames)
    dw, keep = device_weights(hip, binding, dev, w)
    got, plain = _stage(hip, binding, dev, w, dw, latent, frames, 2)
    assert np.all(np.isfinite(plain))
    # an inner value of 3e4 is known to 4e-3, its sine's square to 8e-3, and counts 1e-4 times: below the sums' rounding
    assert f32_err(got, plain) <= 2e-5


def test_unit_with_a_weight_that_cannot_be_split(hip, binding, dev, oracle):
    """3.4e38 in the last unit's k = 1 weights: the tiles are redone as F32 sums,
    the other output channels stay within F32 rounding of the unit without it."""
    frames, row = 7, 11
    w = Weights(binding, 60)
    latent = oracle.gaussian(64 * frames, 8).reshape(64, frames)
    dw, keep = device_weights(hip, binding, dev, w)
    before = _decode(hip, dev, dw, latent, frames, True)
    w.stages[4]["res"][2]["conv1"][0][row, 5, 0] = np.float32(3.4e38)
    dw, keep = device_weights(hip, binding, dev, w)
    after = _decode(hip, dev, dw, latent, frames, True)
    others = np.arange(128) != row
    assert f32_err(after[others], before[others]) <= 1e-5
    assert not np.any(np.isnan(after)) and np.mean(np.abs(after[row]) > 1e30) > 0.99


def test_unit_with_products_that_overflow(hip, binding, dev, oracle):
    """1e25 in a channel between the last unit's convolutions, 1e20 against it in
    a row of the k = 1 weights: that row is infinite, with the sign of the
    product, the other rows stay within F32 rounding of 1e25 times their weight."""
    frames, row = 7, 11
    w = Weights(binding, 61)
    latent = oracle.gaussian(64 * frames, 9).reshape(64, frames)
    unit = w.stages[4]["res"][2]
    unit["conv0"][1][5] = np.float32(1.0037e25)
    dw, keep = device_weights(hip, binding, dev, w)
    before = _decode(hip, dev, dw, latent, frames, True)
    assert np.all(np.isfinite(before))
    for sign in (1, -1):
        unit["conv1"][0][row, 5, 0] = np.float32(sign * 1.0021e20)
        dw, keep = device_weights(hip, binding, dev, w)
        after = _decode(hip, dev, dw, latent, frames, True)
        assert np.all(np.isinf(after[row])) and np.all(np.sign(after[row]) == sign)
        others = np.arange(128) != row
        assert f32_err(after[others], before[others]) <= 1e-5


def _stage(hip, binding, dev, w, dw, latent, frames, s):
    """Stage s (from 0) as the decode computes it, and from the decode's output of
    the stage before by the public upsampler and residual units (F32)."""
    import torch
    nbytes = hip.vae_decode_workspace_bytes(frames)
    ws = torch.full((nbytes // 4,), float("nan"), device=dev)
    audio = torch.empty(2, 1920 * frames, device=dev)
    ci, c, stride = binding.VAE_IN_WIDTH[s], binding.VAE_OUT_WIDTH[s], binding.VAE_STRIDES[s]
    t_in = frames * int(np.prod(binding.VAE_STRIDES[:s]))
    t = t_in * stride
    outputs = [None] * 5
    outputs[s - 1], outputs[s] = torch.empty(ci, t_in, device=dev), torch.empty(c, t, device=dev)
    hip.vae_decode(dw, to_dev(latent, dev), frames, audio, ws, nbytes, stage_outputs=outputs)
    stage = dw.stage[s]
    x, y, h = (torch.empty(c, t, device=dev) for _ in range(3))
    hip.snake_conv_transpose1d(outputs[s - 1], ci, t_in, stage.upsample.weight, c, stride,
                               alpha_log=stage.activation.alpha_log, beta_log=stage.activation.beta_log,
                               bias=stage.upsample.bias, padding=(stride + 1) // 2, y=x)
    for unit, dil in zip(stage.residual, (1, 3, 9)):
        hip.vae_residual_unit(x, c, t, unit, dil, y, h)
        x, y = y, x
    torch.cuda.synchronize()
    return from_dev(outputs[s]), from_dev(x)


@pytest.mark.parametrize("what", ["x nan", "h inf", "h large", "x large", "w0 inf", "w0 nan", "w0 3.4e38", "w1 inf", "w1 nan"])
def test_unit_special_values(hip, binding, dev, oracle, what):
    """A NaN in the latent, infinite and very large (sine arguments beyond the
    reduced form's) inputs and inner values, weights that are not finite: the
    infinities and NaN of the F32 units, the other values to their rounding."""
    frames = 9
    w = Weights(binding, 70)
    latent = oracle.gaussian(64 * frames, 11).reshape(64, frames)
    unit = w.stages[4]["res"][1]
    where, value = what.split()
    if what == "x nan":
        w.stages[4]["res"][0]["conv1"][1][3] = np.nan  # a channel of the second unit's input
    elif what == "x large":
        w.stages[4]["res"][0]["conv1"][1][::9] = np.float32(3e4)
        unit["conv0"][0][:, ::9] *= np.float32(1e-4)
    elif where == "h":
        unit["conv0"][1][::9] = np.float32({"inf": np.inf, "large": 3e4}[value])
        unit["conv1"][0][:, ::9] *= np.float32(1e-4)
    else:
        unit["conv" + where[1]][0][17, 5, 0] = np.float32(value)
    dw, keep = device_weights(hip, binding, dev, w)
    got, plain = _stage(hip, binding, dev, w, dw, latent, frames, 4)
    nan = np.isnan(plain)
    assert np.array_equal(np.isnan(got), nan)
    inf = np.isinf(plain)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(np.sign(got[inf]), np.sign(plain[inf]))
    assert np.any(nan | inf) == (value not in ("large", "3.4e38"))
    ok = np.isfinite(plain)
    if np.any(ok):
        # two F32 sums of 896 and 128 terms, three units: at the scale of their terms
        scale = {"large": 3e4, "3.4e38": np.max(np.abs(plain[ok]))}.get(value, np.maximum(np.abs(plain[ok]), 1.0))
        assert np.max(np.abs(got[ok].astype(np.float64) - plain[ok]) / scale) <= 2e-5


def test_nan_costs_no_more_than_numbers(hip, binding, dev, oracle):
    """A decode of a latent with a NaN (in the end all of the audio): within twice
    the time of an ordinary one, as the F32 launches took the same for both."""
    import torch
    frames = 64
    w = Weights(binding, 80)
    dw, keep = device_weights(hip, binding, dev, w)
    nbytes = hip.vae_decode_workspace_bytes(frames)
    ws = torch.empty(nbytes // 4, device=dev)
    audio = torch.empty(2, 1920 * frames, device=dev)
    latent = to_dev(oracle.gaussian(64 * frames, 12).reshape(64, frames), dev)
    odd = latent.clone()
    odd[7, 5::11] = float("nan")
    times = {}
    for name, x in (("numbers", latent), ("nan", odd)):
        best = 1e9
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            hip.vae_decode(dw, x, frames, audio, ws, nbytes)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times[name] = best
    assert torch.isnan(audio).all()
    assert times["nan"] <= 2 * times["numbers"], times


@pytest.mark.parametrize("xs,ws", [(-112, 0), (0, -112), (-70, -55), (-125, 0)])
@pytest.mark.parametrize("kw,direct", [(7, True), (7, False), (2, True), (1, False)])
def test_tiny_operands(hip, dev, oracle, kw, direct, xs, ws):
    """Inputs or weights (or their products) that are all so small that the parts
    would lose bits: as close to the exact sums as the F32 launch, in the 2-norm
    relative to them (10 % and the smallest F32 steps allowed)."""
    c, c_out, t, stride = (256, 256, 20000, 1) if kw != 2 else (512, 256, 4300, 4)
    if kw == 2:
        x, w, _, _, _ = _t_case(oracle, c, c_out, t, stride, 41)
    else:
        x, w, _, _, _, _ = _case(oracle, c, c_out, t, kw, 41)
    x, w = x * np.float32(2.0 ** xs), w * np.float32(2.0 ** ws)
    n = _direct_floats(c, c_out * stride, kw, t + 1) if direct else -1
    if kw == 2:
        got, plain = _run_t(hip, dev, x, w, None, 4, 2, ws_floats=n), _run_t(hip, dev, x, w, None, 4, 2, split=False)
    else:
        got, plain = (_run(hip, dev, x, w, None, kw // 2, 1, ws_floats=m) for m in (n, None))
    rows = np.arange(0, c_out, 16)
    exact = (_f64_transpose_rows(oracle, x, w, None, 4, 2, None, None, rows) if kw == 2 else
             _f64_rows(oracle, x, w, None, kw // 2, 1, None, None, None, rows))
    scale = 2.0 ** -(xs + ws)  # the sums of squares would underflow
    err = lambda y: np.linalg.norm((y[rows].astype(np.float64) - exact) * scale)
    assert err(got) <= 1.1 * err(plain) + c * kw * 2.0 ** -149 * scale * np.sqrt(exact.size)


@pytest.mark.parametrize("c_in,c_out,kw,dil,t,stride,big", [
    (1024, 1024, 1, 1, 573, 0, False), (2048, 512, 1, 1, 1146, 0, False), (512, 512, 3, 1, 763, 0, False),
    (256, 256, 7, 9, 3120, 0, True), (256, 256, 7, 1, 2616, 0, True), (2048, 1024, 2, 1, 50, 10, True),
    (2048, 1024, 2, 1, 100, 10, True), (512, 512, 7, 3, 15121, 0, True), (1024, 1024, 7, 9, 2520, 0, True),
    (2048, 1024, 2, 1, 1000, 10, True)])
def test_route_is_the_faster_one(hip, dev, oracle, c_in, c_out, kw, dil, t, stride, big):
    """The form that the estimates choose, in the queried workspace or a large
    one, against the F32 launch with its four splits, which the same call takes
    where the workspace meets a tensor past the partial sums (here the bias):
    no slower, within 10 % for the clock and what the estimates cannot see."""
    import torch
    rows = c_out * max(stride, 1)
    cols = t + 1 if stride else t
    n = 4 * rows * ((cols + 3) // 4 * 4)
    n = n + 100_000_000 if big else n
    ws = torch.zeros(n + c_out, device=dev)
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(c_in, t, device=dev, generator=g)
    w = torch.randn(rows * c_in * kw, device=dev, generator=g) * 0.02
    params = dict(alpha_log=torch.zeros(c_in, device=dev), beta_log=torch.zeros(c_in, device=dev))
    pad = (stride + 1) // 2 if stride else dil * (kw - 1) // 2
    y = torch.empty((c_out, (t + 1) * stride - 2 * pad if stride else t), device=dev)

    def call(floats):
        kwargs = dict(workspace=ws, workspace_floats=floats, bias=ws[n:], padding=pad, y=y, **params)
        if stride:
            hip.snake_conv_transpose1d_split(x, c_in, t, w, c_out, stride, **kwargs)
        else:
            hip.snake_conv1d_split(x, c_in, t, w, c_out, kw, dilation=dil, **kwargs)

    best = {n: 1e9, n + c_out: 1e9}
    for _ in range(8):
        for floats in best:
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                call(floats)
            b.record()
            b.synchronize()
            best[floats] = min(best[floats], a.elapsed_time(b) / 5)
    assert best[n] <= 1.1 * best[n + c_out], best
