"""Tiles of 32 and 48 rows with unscaled weights (gemm_rows.hip), at the edges of their row counts, with one to seven K splits (the last arrival adds four
at a time) and with a shorter last one, against float64.  tests/test_plans.py pins that these problems run there."""
import pytest
import torch

from test_gpu_kq_heights import _layer, _rel, _run, workspace  # noqa: F401

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
# (m, k, n, dtype, fmt, group, act_order): (m-blocks, splits, units of 128 K rows per split) of the plan
ROWS = {
    (17, 14336, 4096, BF16, "uint4", 128, False): (2, 4, 28),
    (32, 14336, 4096, BF16, "uint4", 256, False): (2, 4, 28),
    (33, 14336, 4096, F16, "uint4", 128, False): (3, 4, 28),
    (48, 14336, 4096, BF16, "uint4b8", 128, True): (3, 4, 28),
    (48, 18944, 3584, F16, "uint4b8", 128, False): (3, 4, 37),
    (20, 18944, 3648, BF16, "uint4", -1, False): (2, 4, 37),
    (31, 28672, 4096, F16, "uint4b8", -1, False): (2, 4, 56),
    (17, 28672, 4096, F16, "uint4b8", 128, False): (2, 4, 56),
    (29, 18944, 3584, F16, "uint4", -1, False): (2, 4, 37),
    (47, 13824, 5120, BF16, "uint4", 128, False): (3, 3, 36),
    (48, 4096, 11008, F16, "uint4", 128, False): (3, 1, 32),
    (40, 4096, 11008, BF16, "uint4b8", -1, False): (3, 1, 32),
    (37, 5120, 13824, F16, "uint4b8", 128, False): (3, 1, 40),
    # the last split is shorter
    (37, 11008, 4096, BF16, "uint4", 128, False): (3, 4, 22),
    (48, 8064, 6400, BF16, "uint4b8", -1, False): (3, 2, 32),
    (17, 9344, 7168, BF16, "uint4", 128, False): (2, 2, 37),
    (32, 25472, 3072, F16, "uint4b8", 128, False): (2, 5, 40),
    (48, 24192, 3072, BF16, "uint4b8", 128, True): (3, 5, 38),
    (17, 20736, 2304, F16, "uint4", -1, False): (2, 7, 24),
    (33, 18560, 2304, BF16, "uint4", 128, False): (3, 7, 21),
}


def _exact(k, n, fmt, group, dtype, act_order, dev):
    """What _layer's weights are before they are rounded to 16 bits, in float64."""
    from vllm_amd.marlin_utils_test import quantize_weights
    from vllm_amd.scalar_type import scalar_types as st
    g = torch.Generator(device=dev).manual_seed(0)
    w = (torch.randn(k, n, generator=g, device=dev) * 0.02).to(dtype)
    gs = k if group == -1 else group
    _, q, s, z = quantize_weights(w, (st.uint4, st.uint4b8)[fmt == "uint4b8"], gs, zero_points=fmt == "uint4", rule="absmax")
    zero = 8 if z is None else z.double().repeat_interleave(gs, 0)
    ref = (q.double() - zero) * s.double().repeat_interleave(gs, 0)
    if act_order:
        order = torch.randperm(k, generator=g, device=dev)
        by_row = torch.empty_like(order)
        by_row[order] = torch.arange(k, device=dev)
        ref = ref[by_row]
    return ref


@pytest.mark.parametrize("m,k,n,dtype,fmt,group,act_order", list(ROWS))
def test_against_float64(dev, workspace, m, k, n, dtype, fmt, group, act_order):  # noqa: F811
    print(f"rows m={m} k={k} n={n} {dtype} {fmt} group={group} act_order={act_order}", flush=True)
    from vllm_amd.marlin_utils import marlin_permute_bias
    # rounding the result to 11 / 8 bits (rms 2^-11 / sqrt(3) of a binade's mean, 2.1e-4 and 1.66e-3) and fp32 sums on offset weights
    bound = 2.3e-4 if dtype == F16 else 1.75e-3
    layer = _layer(k, n, fmt, group, dtype, act_order, dev)
    exact = _exact(k, n, fmt, group, dtype, act_order, dev)
    g = torch.Generator(device=dev).manual_seed(m)
    a = torch.randn(m, k + 64, generator=g, device=dev).to(dtype)[:, 32:32 + k]  # a strided view
    ref = a.double() @ exact
    out = _run(a, layer, n, k, workspace)
    assert _rel(out, ref) < bound
    assert torch.equal(out, _run(a.contiguous(), layer, n, k, workspace))
    bias = torch.randn(n, generator=g, device=dev).to(dtype)
    assert _rel(_run(a, layer, n, k, workspace, marlin_permute_bias(bias)), ref + bias.double()) < bound
    assert int(workspace.abs().sum()) == 0
    # a row with one element shows the weights themselves, rounded once
    one = torch.zeros(m, k, dtype=dtype, device=dev)
    one[torch.arange(m), torch.arange(m) * 97 % k] = 1
    out = _run(one, layer, n, k, workspace)
    assert torch.equal(out, exact[torch.arange(m, device=dev) * 97 % k].to(dtype))


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_rows_are_independent(dev, workspace, value):  # noqa: F811
    m, k, n = 37, 14336, 4096
    layer = _layer(k, n, "uint4", 128, BF16, False, dev)
    a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(3), device=dev).to(BF16)
    clean = _run(a, layer, n, k, workspace)
    a[36, 5000] = value
    out = _run(a, layer, n, k, workspace)
    assert torch.equal(out[:36], clean[:36]) and not torch.isfinite(out[36]).any()
