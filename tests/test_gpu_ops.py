"""Parity of the stateless operators bf_cuda_gemm_f32 / bf_cuda_conv2d_f32.

Cases follow the reference's own GPU operator test (tests/test_cuda_ops.cu):
the 19x23->17 ReLU GEMM, a strided conv, a 5x5/s4 conv with Inf/NaN injected,
a 2x2/s2 transposed conv and a 1 048 561-row grid (65 536 row tiles), all with
its pattern() fill, plus the stage-1 QKV linear 11264x96 -> 288.

Two references per case:
  * the fp32 CPU oracle / float64 restatement of the operator, held to the
    bf16 tolerance of tests/util.py;
  * the same float64 sum over bf16-rounded operands, held to 1e-5 relative:
    it isolates the kernel's indexing from bf16 input rounding, so a wrong
    tap, row or channel cannot hide inside the bf16 tolerance.
"""

import numpy as np
import pytest

import convref
from util import assert_close, bf16_round, pattern

pytestmark = pytest.mark.gpu


def _t(a, device):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(device)


def _tight(actual, expected, name, rtol=1e-5):
    a = np.asarray(actual, np.float64).ravel()
    e = np.asarray(expected, np.float64).ravel()
    fin = np.isfinite(e)
    scale = np.sqrt(np.mean(e[fin] ** 2)) + 1e-30
    err = np.max(np.abs(a[fin] - e[fin])) / scale
    assert err <= rtol, f"{name}: bf16-operand residual {err:.3e} > {rtol:.1e}"


def run_conv(device, fields, inject_special=False):
    import bfhip
    d = bfhip.ConvDesc(*fields)
    n_in = d.batches * d.input_channels * d.input_height * d.input_width
    n_w = d.input_channels * d.output_channels * d.kernel_height * d.kernel_width
    x = pattern(np.arange(n_in)).reshape(d.batches, d.input_channels, d.input_height,
                                         d.input_width)
    if d.transpose:
        w = (pattern(np.arange(n_w) + 11) * np.float32(0.1)).reshape(
            d.input_channels, d.output_channels, d.kernel_height, d.kernel_width)
    else:
        w = (pattern(np.arange(n_w) + 11) * np.float32(0.1)).reshape(
            d.output_channels, d.input_channels, d.kernel_height, d.kernel_width)
    b = pattern(np.arange(d.output_channels) + 29) * np.float32(0.2)
    if inject_special:
        x.reshape(-1)[0] = np.inf
        w.reshape(-1)[0] = 0.0
        x.reshape(-1)[-1] = np.nan
    import torch
    out = torch.empty((d.batches, d.output_channels, d.output_height, d.output_width),
                      device=device)
    xt, wt, bt = _t(x, device), _t(w, device), _t(b, device)
    ok, msg = bfhip.conv2d_raw(d, xt.data_ptr(), wt.data_ptr(), bt.data_ptr(), out.data_ptr())
    assert ok, msg
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    return d, x, w, b, got


CONV_CASES = {
    # fields: batches, Ci, Co, IH, IW, KH, KW, SH, SW, PH, PW, OH, OW, transpose, relu
    "stride": ((2, 3, 5, 6, 7, 3, 3, 2, 2, 1, 1, 3, 4, 0, 1), False),
    "wide_inf_nan": ((1, 2, 3, 9, 10, 5, 5, 4, 4, 2, 2, 3, 3, 0, 0), True),
    "transpose": ((1, 3, 5, 4, 6, 2, 2, 2, 2, 0, 0, 8, 12, 1, 1), False),
    "large_grid": ((1, 1, 1, 1, 1048561, 1, 1, 1, 1, 0, 0, 1, 1048561, 0, 0), False),
    "k3_c64_relu": ((2, 64, 96, 13, 17, 3, 3, 1, 1, 1, 1, 13, 17, 0, 1), False),
    "k5_s2_odd": ((1, 7, 33, 21, 19, 5, 5, 2, 2, 2, 2, 11, 10, 0, 0), False),
}


@pytest.mark.parametrize("case", sorted(CONV_CASES))
def test_conv_reference_cases(device, case):
    fields, special = CONV_CASES[case]
    d, x, w, b, got = run_conv(device, fields, special)
    expected = convref.conv_abi(d, x, w, b)
    assert_close(got, expected, case)
    _tight(got, convref.conv_abi(d, x, w, b, round_inputs=bf16_round), case)


def test_conv_matches_oracle(device):
    """Strided conv with bias against the CPU oracle (oracle port, OpenMP)."""
    import oracle
    import bfhip
    rng = np.random.default_rng(3)
    x = rng.standard_normal((2, 16, 20, 24)).astype(np.float32)
    w = (rng.standard_normal((40, 16, 3, 3)) / 12).astype(np.float32)
    b = rng.standard_normal(40).astype(np.float32)
    ref = oracle.Oracle("port").conv2d(x, w, b, stride=(2, 2), pad=(1, 1))
    got = bfhip.conv2d_f32(_t(x, device), _t(w, device), _t(b, device), stride=(2, 2),
                           padding=(1, 1)).cpu().numpy()
    assert_close(got, ref, "conv vs oracle")


def test_conv_transpose_matches_oracle(device):
    import oracle
    import bfhip
    rng = np.random.default_rng(4)
    x = rng.standard_normal((1, 6, 5, 7)).astype(np.float32)
    w = (rng.standard_normal((6, 10, 2, 2)) / 3).astype(np.float32)  # IOHW
    b = rng.standard_normal(10).astype(np.float32)
    ref = oracle.Oracle("port").conv_transpose2d(x, w, b, stride=(2, 2))
    got = bfhip.conv2d_f32(_t(x, device), _t(w, device), _t(b, device), stride=(2, 2),
                           transpose=True).cpu().numpy()
    assert_close(got, ref, "transposed conv vs oracle")


def test_gemm_reference_fixture(device):
    """test_cuda_ops.cu:118-153: 19x23 -> 17, bias, ReLU, pattern() fill."""
    import bfhip
    rows, k, n = 19, 23, 17
    a = pattern(np.arange(rows * k)).reshape(rows, k) * np.float32(0.2)
    w = pattern(np.arange(n * k) + 7).reshape(n, k) * np.float32(0.1)
    b = pattern(np.arange(n) + 3)
    got = bfhip.gemm_f32(_t(a, device), _t(w, device), _t(b, device), relu=True).cpu().numpy()
    assert_close(got, convref.gemm_abi(a, w, b, True), "gemm 19x23x17")
    _tight(got, convref.gemm_abi(a, w, b, True, round_inputs=bf16_round), "gemm 19x23x17")


def test_gemm_config1_matches_oracle(device):
    """X[11264x96] W[288x96] + bias, ~N(0,1)/sqrt(96), seed 0."""
    import oracle
    import bfhip
    from bfhip import bfw
    x = bfw.randn(0, "config1.x", (11264, 96), 1 / np.sqrt(96))
    w = bfw.randn(0, "config1.w", (288, 96), 1 / np.sqrt(96))
    b = bfw.randn(0, "config1.b", (288,), 1 / np.sqrt(96))
    ref = oracle.Oracle("port").linear(x, w, b)
    got = bfhip.gemm_f32(_t(x, device), _t(w, device), _t(b, device)).cpu().numpy()
    assert_close(got, ref, "config1 linear")
    _tight(got, convref.gemm_abi(x, w, b, False, round_inputs=bf16_round), "config1 linear")


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 5, 4), (300, 96, 96), (129, 130, 131),
                                   (1000, 384, 1536), (64, 3072, 768), (513, 8, 33),
                                   (200, 96, 145), (77, 31, 250), (33, 64, 288)])
def test_gemm_shapes(device, shape):
    import bfhip
    m, k, n = shape
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    got = bfhip.gemm_f32(_t(x, device), _t(w, device), _t(b, device)).cpu().numpy()
    assert_close(got, convref.gemm_abi(x, w, b, False), f"gemm {shape}")
    _tight(got, convref.gemm_abi(x, w, b, False, round_inputs=bf16_round), f"gemm {shape}")


def test_gemm_unaligned_operands(device):
    """Row pitch not a multiple of 4 floats and offset base pointers (scalar path)."""
    import bfhip
    import torch
    rng = np.random.default_rng(9)
    x = rng.standard_normal((50, 31)).astype(np.float32)
    w = rng.standard_normal((20, 31)).astype(np.float32)
    xt = torch.zeros(50 * 31 + 1, device=device)
    xt[1:] = _t(x, device).reshape(-1)
    xv = xt[1:].view(50, 31)
    got = bfhip.gemm_f32(xv, _t(w, device)).cpu().numpy()
    _tight(got, convref.gemm_abi(x, w, None, False, round_inputs=bf16_round), "unaligned")


def test_repeat_is_bit_exact(device):
    """Determinism gate (reference test_cuda_camera_full.cu:69-72): no atomics."""
    import bfhip
    rng = np.random.default_rng(5)
    x = _t(rng.standard_normal((4096, 384)), device)
    w = _t(rng.standard_normal((1152, 384)) / 20, device)
    a = bfhip.gemm_f32(x, w).cpu().numpy()
    b = bfhip.gemm_f32(x, w).cpu().numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _gemm_route(*args):
    """GemmRoute (ops.hip) of a call: asserted, so that a case keeps running the
    kernel it is there for."""
    from test_launch_limits import gemm_route
    return gemm_route(*args)


# (rows, in, out, relu, bias, inject Inf/NaN): shapes the short-reduction
# panel kernel is chosen for (K <= 128, K % 4 == 0, 144 < N <= 288, N % 4 == 0):
# ragged row panels (1, 7, 63 and 65 rows in the last), N not a multiple of 16,
# K not a multiple of 8 or 32, one to four 32-deep k-steps, ReLU, no bias, and
# Inf/NaN operands.
PANEL_CASES = [(10241, 100, 148, True, True, False), (4039, 4, 160, False, False, False),
               (9023, 128, 200, False, True, False), (10305, 32, 288, True, True, True),
               (11264, 96, 288, False, True, False), (8385, 60, 252, False, True, False),
               (12353, 124, 244, True, False, True), (4161, 36, 204, False, False, True)]


@pytest.mark.parametrize("case", PANEL_CASES)
def test_gemm_panel_equals_tiled_core(device, case):
    """The panel kernel (aligned operands) against the tiled core, reached by
    handing the library an output that is not 16-byte aligned: same bf16
    operand rounding, same 32-deep k order and bias after the accumulation,
    so the two must agree bit for bit; and both within 1e-5 of the float64
    sum over bf16-rounded operands."""
    import bfhip
    import torch
    m, k, n, relu, with_bias, special = case
    print(f"[case] panel gemm {m}x{k}->{n} relu={relu} bias={with_bias} special={special}",
          flush=True)
    assert _gemm_route(m, k, n) == 6
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32) if with_bias else None
    if special:
        x[0, 0] = np.inf
        x[-1, -1] = np.nan
    xt, wt = _t(x, device), _t(w, device)
    bt = _t(b, device) if with_bias else None
    panel = bfhip.gemm_f32(xt, wt, bt, relu=relu)
    buf = torch.empty(m * n + 1, device=device)
    tiled_out = buf[1:].view(m, n)
    assert bfhip.hip_lib().bfhip_gemm_route(4096, 4096, None, 4100, m, k, n) not in (3, 6)
    bfhip.gemm_f32(xt, wt, bt, relu=relu, out=tiled_out)
    torch.cuda.synchronize()
    a, t = panel.cpu().numpy(), tiled_out.cpu().numpy()
    assert np.array_equal(a.view(np.uint32), t.view(np.uint32)), "panel and tiled core differ"
    want = convref.gemm_abi(x, w, b, relu, round_inputs=bf16_round)
    if special:
        assert np.array_equal(np.isnan(a), np.isnan(want)) and np.array_equal(np.isinf(a), np.isinf(want))
    _tight(a, want, f"panel gemm {case}")


# Fields as CONV_CASES.  Shapes at the edges of the direct kernel's tiles and
# channel blocks: one channel; blocks of 32 with one channel over, one under
# and seven short; whole and ragged output-channel tiles (33, 129); kernels
# taller than wide; 36 taps (the most it takes) and 49 (the gather core's);
# padding wider than the kernel's reach; a stride that leaves one pixel per
# patch row; an output larger and one smaller than the input defines; more
# than one column tile and image; a flat 1x1 with an odd pixel count;
# transposed 2x2 on odd widths, 3x3 and 1x3 kernels, and a padded one (the
# gather core's).
DIRECT_CASES = {
    "one_channel": (2, 1, 33, 9, 11, 3, 3, 1, 1, 1, 1, 9, 11, 0, 1),
    "tail_33": (1, 33, 40, 12, 20, 3, 3, 1, 1, 1, 1, 12, 20, 0, 0),
    "tail_31_vec": (1, 60, 129, 17, 23, 3, 3, 1, 1, 1, 1, 17, 23, 0, 1),
    "tail_25": (3, 25, 64, 7, 50, 3, 3, 2, 2, 1, 1, 4, 25, 0, 0),
    "tall": (1, 12, 20, 15, 14, 5, 2, 1, 2, 2, 0, 15, 7, 0, 0),
    "taps_36": (1, 9, 17, 14, 13, 6, 6, 1, 1, 2, 3, 13, 14, 0, 0),
    "taps_49": (1, 9, 17, 14, 13, 7, 7, 1, 1, 3, 3, 14, 13, 0, 0),
    "wide_pad": (1, 8, 16, 6, 5, 3, 3, 1, 1, 4, 5, 12, 13, 0, 0),
    "stride_7": (1, 20, 24, 40, 50, 3, 3, 7, 9, 1, 1, 6, 6, 0, 1),
    "larger_out": (1, 16, 16, 8, 8, 3, 3, 1, 1, 1, 1, 11, 10, 0, 0),
    "smaller_out": (2, 16, 16, 9, 9, 3, 3, 1, 1, 1, 1, 5, 4, 0, 0),
    "full_tiles": (2, 64, 256, 32, 88, 3, 3, 1, 1, 1, 1, 32, 88, 0, 1),
    "flat_odd": (2, 70, 45, 9, 31, 1, 1, 1, 1, 0, 0, 9, 31, 0, 0),
    "flat_vec": (2, 68, 130, 12, 30, 1, 1, 1, 1, 0, 0, 12, 30, 0, 1),
    "strided_1x1": (1, 24, 40, 13, 18, 1, 1, 2, 3, 0, 0, 7, 6, 0, 0),
    "up_2x2_odd": (2, 37, 19, 5, 7, 2, 2, 2, 2, 0, 0, 10, 14, 1, 1),
    "up_2x2_vec": (1, 40, 66, 10, 12, 2, 2, 2, 2, 0, 0, 20, 24, 1, 0),
    "up_3x3": (1, 10, 5, 6, 8, 3, 3, 3, 3, 0, 0, 18, 24, 1, 0),
    "up_1x3": (1, 10, 8, 6, 8, 1, 3, 1, 3, 0, 0, 6, 24, 1, 0),
    "up_padded": (1, 10, 8, 6, 8, 2, 2, 2, 2, 1, 1, 10, 14, 1, 0),
}


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("case", sorted(DIRECT_CASES))
def test_conv_direct_edges(device, case, special):
    """Against the float64 sum over bf16-rounded operands (1e-5 of the RMS:
    fp32 sums of at most 576 products), with and without Inf / NaN inputs,
    which may reach only the sums they belong to."""
    print(f"[case] conv {case} special={special}", flush=True)
    d, x, w, b, got = run_conv(device, DIRECT_CASES[case], special)
    want = convref.conv_abi(d, x, w, b, round_inputs=bf16_round)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    _tight(got, want, case)


# (route, fields as CONV_CASES): every kernel at odd sizes, asserted to be the
# one that runs (ConvRoute, + 8 with float4 weights, + 16 with float4 patches):
# the direct tiles 128 x 160 (0), 64 x 128 (1), 32 x 64 (2) and 32 x 32 (3),
# plain and transposed, and the gather core (4) with one, two and four blocks of
# 32 output channels per tile, by its choice (few channels), by its taps and as
# the padded transposed layers that only it takes.
CONV_ROUTE_CASES = [
    (0, (4, 16, 203, 116, 36, 1, 1, 1, 1, 0, 0, 116, 36, 0, 1)),
    (0, (3, 17, 132, 21, 194, 3, 3, 1, 1, 1, 1, 21, 194, 0, 0)),
    (8, (4, 92, 134, 105, 26, 1, 1, 1, 1, 0, 0, 105, 26, 0, 1)),
    (8, (2, 2, 88, 115, 149, 6, 6, 1, 1, 3, 3, 116, 150, 0, 0)),
    (24, (2, 28, 193, 105, 80, 1, 1, 1, 1, 0, 0, 105, 80, 0, 0)),
    (8, (2, 85, 9, 107, 157, 2, 2, 2, 2, 0, 0, 214, 314, 1, 0)),
    (24, (2, 33, 19, 105, 180, 2, 2, 2, 2, 0, 0, 210, 360, 1, 1)),
    (1, (2, 1, 239, 31, 73, 1, 1, 1, 1, 0, 0, 31, 73, 0, 1)),
    (9, (2, 44, 157, 53, 125, 1, 1, 1, 1, 0, 0, 53, 125, 0, 0)),
    (25, (2, 60, 43, 110, 120, 1, 1, 1, 1, 0, 0, 110, 120, 0, 1)),
    (9, (3, 1, 107, 41, 31, 2, 2, 2, 2, 0, 0, 82, 62, 1, 1)),
    (25, (3, 1, 188, 10, 68, 2, 2, 2, 2, 0, 0, 20, 136, 1, 0)),
    (2, (2, 2, 4, 59, 95, 1, 1, 1, 1, 0, 0, 59, 95, 0, 0)),
    (10, (3, 12, 5, 49, 157, 1, 1, 1, 1, 0, 0, 49, 157, 0, 1)),
    (26, (2, 4, 7, 52, 85, 1, 1, 1, 1, 0, 0, 52, 85, 0, 0)),
    (2, (3, 4, 103, 15, 55, 2, 2, 2, 2, 0, 0, 30, 110, 1, 1)),
    (10, (2, 1, 18, 41, 35, 2, 2, 2, 2, 0, 0, 82, 70, 1, 0)),
    (26, (3, 1, 10, 73, 20, 2, 2, 2, 2, 0, 0, 146, 40, 1, 1)),
    (3, (1, 2, 4, 5, 7, 1, 1, 2, 2, 0, 0, 3, 4, 0, 0)),
    (11, (3, 20, 4, 5, 5, 1, 1, 2, 2, 0, 0, 3, 3, 0, 1)),
    (27, (2, 4, 5, 6, 10, 1, 1, 1, 1, 0, 0, 6, 10, 0, 0)),
    (3, (1, 264, 5, 51, 4, 2, 2, 2, 2, 0, 0, 102, 8, 1, 0)),
    (11, (2, 1, 7, 5, 5, 2, 2, 2, 2, 0, 0, 10, 10, 1, 1)),
    (27, (1, 1, 4, 4, 6, 2, 2, 2, 2, 0, 0, 8, 12, 1, 0)),
    (4, (2, 1, 14, 65, 183, 1, 1, 1, 1, 0, 0, 65, 183, 0, 1)),
    (4, (2, 1, 28, 127, 89, 2, 2, 2, 2, 0, 0, 254, 178, 1, 0)),
    (4, (1, 9, 33, 14, 13, 7, 7, 1, 1, 3, 3, 14, 13, 0, 0)),
    (4, (2, 5, 65, 19, 11, 7, 7, 2, 2, 3, 3, 10, 6, 0, 1)),
    (4, (1, 11, 129, 12, 15, 7, 7, 1, 1, 3, 3, 12, 15, 0, 0)),
    (4, (2, 10, 33, 6, 8, 2, 2, 2, 2, 1, 1, 10, 14, 1, 1)),
    (4, (1, 12, 129, 5, 7, 3, 3, 2, 2, 1, 1, 9, 13, 1, 0)),
]


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("route,fields", CONV_ROUTE_CASES)
def test_conv_each_kernel(device, route, fields, special):
    """As test_conv_direct_edges (sums of at most 1452 products)."""
    import bfhip
    from test_launch_limits import conv_route
    print(f"[case] conv {fields} special={special}", flush=True)
    assert conv_route(bfhip.ConvDesc(*fields))[0] == route
    d, x, w, b, got = run_conv(device, fields, special)
    want = convref.conv_abi(d, x, w, b, round_inputs=bf16_round)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    _tight(got, want, fields)


def test_conv_unaligned_operands(device):
    """Input, weights and output off the 16-byte grid (scalar fetches, and
    float stores in a transposed layer)."""
    import bfhip
    import torch
    rng = np.random.default_rng(21)
    for shape, wshape, kw in (((1, 32, 12, 16), (48, 32, 3, 3), dict(padding=(1, 1))),
                              ((1, 32, 12, 16), (48, 32, 1, 1), {}),
                              ((1, 32, 12, 16), (32, 24, 2, 2), dict(stride=(2, 2), transpose=True))):
        x, w = _t(rng.standard_normal(shape), device), _t(rng.standard_normal(wshape) / 17, device)
        want = bfhip.conv2d_f32(x, w, **kw)
        off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)  # noqa: E731
        out = off(torch.zeros_like(want))
        bfhip.conv2d_f32(off(x), off(w), out=out, **kw)
        _tight(out.cpu().numpy(), want.cpu().numpy(), f"unaligned conv {wshape}")


# (rows, in, out, relu, bias, inject Inf/NaN): the thin kernel (eight waves
# sharing the reduction, or four short tiles per workgroup) and each tiled
# core at the edges of their tiles and k-blocks, with and without 16-byte rows.
GEMM_EDGE_CASES = [(1, 1, 1, True, True, False), (15, 31, 17, False, True, False),
                   (17, 33, 15, True, False, True), (16, 256, 16, False, False, False),
                   (33, 257, 40, False, True, True), (6, 2386, 4, False, True, False),
                   (7, 1340, 241, True, True, False), (5000, 8, 16, False, True, False),
                   (4097, 7, 3, True, False, False), (300, 512, 513, False, True, False),
                   (999, 130, 1001, False, True, True), (6001, 100, 290, True, True, False),
                   (4225, 200, 1540, False, True, False)]


# The same with the kernel that is to run: each at the edges of its tile and
# k-block, loads of four floats and of one, the PANEL_CASES shapes of few rows.
GEMM_ROUTE_CASES = [(0, (4225, 388, 1540, True, True, False)), (0, (16753, 79, 79, False, True, True)),
                    (1, (6001, 100, 290, True, True, False)), (1, (2865, 337, 277, False, True, True)),
                    (2, (300, 1028, 1021, False, True, False)), (2, (500, 259, 401, True, False, True)),
                    (3, (201, 260, 255, True, True, True)), (3, (6, 2387, 5, False, True, False)),
                    (3, (64, 4, 160, False, False, False)), (3, (5, 128, 200, False, True, False)),
                    (3, (130, 32, 288, True, True, True)), (3, (65, 60, 252, False, True, False)),
                    (4, (17406, 14, 13, True, True, False)), (4, (40190, 142, 1, False, True, True)),
                    (4, (2500, 8, 161, False, False, True)), (2, (1001, 100, 148, True, True, False)),
                    (7, (60715, 64, 12, True, True, True)), (7, (91847, 41, 9, False, True, False)),
                    (8, (82455, 4, 57, True, True, True)), (8, (62014, 31, 57, False, False, False))]


@pytest.mark.parametrize("route,case", GEMM_ROUTE_CASES)
def test_gemm_each_kernel(device, route, case):
    assert _gemm_route(*case[:3]) == route
    test_gemm_edges(device, case)


@pytest.mark.parametrize("case", GEMM_EDGE_CASES)
def test_gemm_edges(device, case):
    """Against the float64 sum over bf16-rounded operands (1e-5 of the RMS, as
    test_gemm_shapes at K = 3072); rows past the last and columns past K must
    not reach a sum, Inf and NaN only their own."""
    import bfhip
    m, k, n, relu, with_bias, special = case
    print(f"[case] gemm {case}", flush=True)
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32) if with_bias else None
    if special:
        x[0, 0] = np.inf
        x[-1, -1] = np.nan
        w[-1, 0] = 0.0
    got = bfhip.gemm_f32(_t(x, device), _t(w, device), _t(b, device) if with_bias else None,
                         relu=relu).cpu().numpy()
    want = convref.gemm_abi(x, w, b, relu, round_inputs=bf16_round)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    _tight(got, want, f"gemm {case}")


def test_gemm_very_many_rows(device):
    """2^30 + 77 rows: tiles of 64 rows would need more threads than a launch
    holds.  One product per element, so the result is exact."""
    import bfhip
    import torch
    m = 2 ** 30 + 77
    x = torch.randn(m, 1, device=device)
    w = torch.full((1, 1), 0.5, device=device)
    out = torch.empty(m, 1, device=device)
    print(f"[case] gemm {m}x1 -> 1", flush=True)
    bfhip.gemm_f32(x, w, out=out)
    for a in range(0, m, 2 ** 28):
        assert torch.equal(out[a:a + 2 ** 28], x[a:a + 2 ** 28].bfloat16().float() * 0.5), a


def test_conv_very_many_pixels(device):
    """1.25 * 2^30 output pixels: more than a launch of the direct kernel holds.
    One product per element, so the result is exact."""
    import bfhip
    import torch
    shape = (20, 1, 8192, 8192)
    x = torch.randn(shape, device=device)
    w = torch.full((1, 1, 1, 1), 0.5, device=device)
    out = torch.empty(shape, device=device)
    print(f"[case] conv 1x1 on {shape}", flush=True)
    bfhip.conv2d_f32(x, w, out=out)
    for n in range(shape[0]):
        assert torch.equal(out[n], x[n].bfloat16().float() * 0.5), n
