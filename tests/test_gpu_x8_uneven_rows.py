"""The 8-bit matrix unit (gemm_x8.hip) on rows with few activations of very different size: columns whose weights at the large ones are zero have
nothing but the small ones to show.  Every result is held to 1.5 * 2^-8 of the sum of its products' magnitudes (a kernel with weights rounded to
bf16 keeps 2 * 2^-8): 2^-8 is the rounding of the result; the unit cuts each of eight neighbouring products at 2^-14 of the largest, counted up to four
times too large where its weight is subnormal, 7 * 2^-12 in the high term and a sixteenth of that in the low one: 0.46 * 2^-8."""
import pytest
import torch

from test_gpu_x8 import LARGE, SPLIT, _layer, _run
from test_gpu_x8_moe import Moe
from test_gpu_x8_prepared import PINNED as PREPARED

pytestmark = pytest.mark.gpu


@pytest.fixture
def workspace(dev):
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    return marlin_make_workspace_new(dev)


def _rows(m, k, dev, seed=1):
    """Rows with all their activations in one step of 128 columns.  Every third: 2^13, and side by side 1 and 2^-12.  The others: 1 to 31, between 1
    and 2^-20 in size."""
    g = torch.Generator(device=dev).manual_seed(seed)
    a = torch.zeros(m, k // 128, 128, device=dev)
    part = torch.ldexp(torch.randn(m, 128, generator=g, device=dev), torch.randint(-20, 1, (m, 128), generator=g, device=dev))
    part *= torch.rand(m, 128, generator=g, device=dev).argsort(-1) < torch.randint(1, 32, (m, 1), generator=g, device=dev)
    for i in range(0, m, 3):
        at = 8 * (i % 16) + i % 7
        part[i] = 0
        part[i, at], part[i, at + 1], part[i, (at + 8) % 128] = 1, 2.0 ** -12, 2.0 ** 13
    r = torch.arange(m, device=dev)
    a[r, r % (k // 128)] = part
    return a.view(m, k).bfloat16()


def _check(out, a, exact):
    assert bool(torch.isfinite(out).all())
    ref, size = a.double() @ exact, a.double().abs() @ exact.abs()
    worst = float(((out.double() - ref).abs() / size.clamp(min=2.0 ** -60)).max())
    assert worst <= 1.5 * 2.0 ** -8, worst


@pytest.mark.parametrize("k,n,m", [LARGE, SPLIT, (1024, 16448, 512)])
@pytest.mark.parametrize("fmt,group", [("uint4b8", 128), ("uint4", 128), ("uint4b8", -1)])
def test_dense(dev, workspace, k, n, m, fmt, group):
    layer = _layer(k, n, fmt, group, dev, seed=6)
    a = _rows(m, k, dev)
    _check(_run(a, layer, n, k, workspace), a, layer[4])


@pytest.mark.parametrize("k,n,m", PREPARED[:2])
def test_prepared_weights(dev, workspace, k, n, m):
    layer = _layer(k, n, "uint4", 128, dev, seed=6)
    a = _rows(m, k, dev)
    _check(_run(a, layer, n, k, workspace), a, layer[4])


@pytest.mark.parametrize("group", [128, -1])
def test_moe_blocks_of_128(dev, group):
    moe = Moe(dev, 1024, 576, [300, 40, 0, 129, 127, 128], group)
    a = _rows(moe.tokens, moe.k, dev)
    out = moe.gemm(a, False)
    for e in range(moe.e):
        mine = moe.ids.flatten() == e
        if bool(mine.any()):
            _check(out[mine], a[mine], moe.exact[e])
