"""Dense bf16 problems with zero points and many rows on the 8-bit matrix unit with prepared weights (gemm_x8.hip: x8_weights_kernel,
x8_prepared_kernel): remainders of rows, columns and K steps, scale groups, exponents, outliers, infinities and NaNs.  Bounds as in
test_gpu_x8.py: the weights stay exact, 1.66e-3 of the root mean square is the rounding of the result."""
import ctypes

import pytest
import torch

from test_gpu_x8 import _c_args, _layer, _rel, _run

pytestmark = pytest.mark.gpu

SHAPES = [(512, 28672, 2040), (256, 8256, 4000), (384, 16448, 2010)]  # (K, N, M); the last strips of the latter two are one n-tile
PINNED = [(512, 28672, 3500), (256, 20544, 4090), (384, 16448, 3060)]  # the same, with prepared weights (test_plans.py); those above run without
WEIGHTS = [(g, shapes[i]) for shapes in (SHAPES, PINNED) for g, i in ((128, 0), (128, 1), (128, 2), (256, 0), (-1, 0), (-1, 1))]
OVER_STATIC = (512, 131072, 2040)  # whose prepared weights exceed the static entry point's buffer


@pytest.fixture
def workspace(dev):
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    return marlin_make_workspace_new(dev)


@pytest.mark.parametrize("group,shape", WEIGHTS)
def test_against_exact_weights(dev, workspace, group, shape):
    from vllm_amd.marlin_utils import marlin_permute_bias
    k, n, m = shape
    layer = _layer(k, n, "uint4", group, dev)
    g = torch.Generator(device=dev).manual_seed(m)
    a = torch.randn(m, k + 64, generator=g, device=dev).bfloat16()[:, 32:32 + k]  # a strided view
    ref = a.double() @ layer[4]
    out = _run(a, layer, n, k, workspace)
    assert _rel(out, ref) < 1.75e-3
    assert torch.equal(out, _run(a.contiguous(), layer, n, k, workspace))
    bias = torch.randn(n, generator=g, device=dev).bfloat16()
    assert _rel(_run(a, layer, n, k, workspace, marlin_permute_bias(bias)), ref + bias.double()) < 1.75e-3


@pytest.mark.parametrize("group,shape", WEIGHTS)
def test_one_hot_rows(dev, workspace, group, shape):
    """Rows +-2^e * (unit vector), e from one end of bf16's exponents to the other: single products, exact to the last bit."""
    k, n, m = shape
    layer = _layer(k, n, "uint4", group, dev, seed=1)
    r = torch.arange(m, device=dev)
    ks, e = (7 * r) % k, (r % 220) - 120
    a = torch.zeros(m, k, device=dev, dtype=torch.bfloat16)
    a[r, ks] = torch.where(r % 2 == 0, 1.0, -1.0).to(dev).mul(torch.ldexp(torch.ones(m, device=dev, dtype=torch.float64), e)).bfloat16()
    ref = a[r, ks].double().unsqueeze(1) * layer[4][ks]
    normal = ref.abs() >= 2.0 ** -118  # (below: fp32 and bf16 subnormals on the way)
    out = _run(a, layer, n, k, workspace)
    assert torch.equal(torch.where(normal, out.double(), 0), torch.where(normal, ref.bfloat16().double(), 0))


@pytest.mark.parametrize("group,shape", WEIGHTS)
def test_special_values_and_outliers(dev, workspace, group, shape):
    """Infinities and NaNs in some rows, in others activations 10^3 .. 10^9 times the others: what the float64 product gives (columns whose
    weight at the outlier is zero are as good as any), and rows without them are untouched."""
    k, n, m = shape
    layer = _layer(k, n, "uint4", group, dev, seed=3)
    g = torch.Generator(device=dev).manual_seed(7)
    plain = torch.randn(m, k, generator=g, device=dev)
    a = plain.clone()
    rows = torch.arange(0, m, 3, device=dev)
    at = torch.randint(0, k, (len(rows),), generator=g, device=dev)
    a[rows, at] *= 10.0 ** (3 + 6 * torch.rand(len(rows), generator=g, device=dev))
    a[4, 5], a[m - 1, k - 1], a[40, 100] = float("inf"), float("-inf"), float("nan")
    a, plain = a.bfloat16(), plain.bfloat16()
    out, clean, ref = _run(a, layer, n, k, workspace), _run(plain, layer, n, k, workspace), a.double() @ layer[4]
    for r in (4, m - 1, 40):
        assert torch.equal(torch.isnan(out[r]), torch.isnan(ref[r]))
        fin = ~torch.isnan(ref[r])
        assert torch.equal(out[r].double()[fin], ref[r][fin])
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[rows] = False
    keep[[4, m - 1, 40]] = False
    assert torch.equal(out[keep], clean[keep])
    rows, at = rows[torch.isfinite(ref[rows]).all(1)], at[torch.isfinite(ref[rows]).all(1)]
    zero = layer[4][at] == 0
    assert int(zero.sum()) > 1000
    assert float((out[rows].double() - ref[rows])[zero].norm() / ref[rows][zero].norm()) < 1.75e-3
    assert _rel(out[rows], ref[rows]) < 1.75e-3


def test_static_entry_point(dev):
    """Prepared weights that fit the library's own buffer, and a problem whose do not, which runs without them."""
    from vllm_amd import _lib
    lib = _lib.load()
    for k, n, m in (SHAPES[1], OVER_STATIC):
        layer = _layer(k, n, "uint4", 128, dev, seed=4)
        a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(9), device=dev).bfloat16()
        c = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
        args = _c_args(_lib, a, c, layer, n, k, k // 128)
        args.wtype, args.b_zeros = _lib.WTYPE_U4, layer[2].data_ptr()
        assert (lib.w4a16_gemm_scratch_bytes(ctypes.byref(args)) > _lib.STATIC_SCRATCH_BYTES) == (n == OVER_STATIC[1])
        assert lib.w4a16_marlin_gemm_static(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)) == 0, lib.w4a16_last_error()
        assert _rel(c, a.double() @ layer[4]) < 2.5e-3
