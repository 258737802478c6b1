"""MoE blocks of 64 slots with integer 4-bit weights on tiles of 256 and 512 columns (gemm_slots.hip): live m-blocks, blocks without a row, last strips of
one n-tile, tiles cut along K, foreign experts, act-order, infinities and NaNs in neighbours of a block, both fused epilogues."""
import pytest
import torch

from test_gpu_group_constants import TYPES, _one_hot
from test_gpu_kq_heights import _layer

pytestmark = pytest.mark.gpu

COUNTS = [64, 1, 16, 17, 0, 32, 33, 48, 49, 100]  # tokens of each expert
# n whose blocks, 10 to 18 at most, are few tiles of 512 columns, and n for which they are more (see test_plans.py)
NARROW, WIDE = 2112, 39360


def _routing(counts, dev, emap=None):
    from vllm_amd.moe_align_block_size import moe_align_block_size
    ids = torch.tensor([x for x, cnt in enumerate(counts) for _ in range(cnt)], dtype=torch.int32, device=dev)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(3)).to(dev)]
    return ids, moe_align_block_size(ids[:, None], 64, len(counts), emap)


def _gemm(a, layers, routing, n, k, dev, act_order=False, foreign=False, weights=None):
    import vllm_amd.ops as ops
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    mq, ms, mz = (torch.stack([layer[i] for layer in layers]) for i in range(3))
    e = torch.empty((len(layers), 0), dtype=torch.int32, device=dev)
    g_idx, perm = (torch.stack([layer[i] for layer in layers]) for i in (3, 4)) if act_order else (e, e)
    s, x, t = routing
    c = torch.full((len(a), n), 7.0, dtype=a.dtype, device=dev)
    return ops.moe_wna16_marlin_gemm(
        a, c, mq, None, ms, None, mz, g_idx, perm, marlin_make_workspace_new(dev, 4), s, x, t,
        torch.ones(len(a), 1, device=dev) if weights is None else weights, moe_block_size=64, top_k=1, mul_topk_weights=weights is not None,
        is_ep=foreign, b_q_type=layers[0][5], size_m=len(a), size_n=n, size_k=k, is_k_full=True, use_atomic_add=False, use_fp32_reduce=True,
        is_zp_float=False)


@pytest.mark.parametrize("dtype,fmt", TYPES)
@pytest.mark.parametrize("group", [32, 64, 128, -1])
@pytest.mark.parametrize("k,n", [(512, NARROW), (256, WIDE)])
def test_one_hot_rows(dev, dtype, fmt, group, k, n):
    """The weights' rows come out as they are, on both widths."""
    layers = [_layer(k, n, fmt, group, dtype, False, dev, seed=i) for i in range(len(COUNTS))]
    ids, routing = _routing(COUNTS, dev)
    a, rows = _one_hot(len(ids), k, dtype, dev)
    out = _gemm(a, layers, routing, n, k, dev)
    assert torch.equal(out, torch.stack([layers[int(i)][-1][r] for i, r in zip(ids, rows)]).to(dtype))


@pytest.mark.parametrize("dtype,fmt,act_order", [t + (False,) for t in TYPES] + [(torch.bfloat16, "uint4b8", True)])
@pytest.mark.parametrize("group", [32, 128, -1])
@pytest.mark.parametrize("n", [NARROW, WIDE])
def test_cut_along_k(dev, dtype, fmt, act_order, group, n):
    """K long enough that tiles are cut: fp32 sums of exact products, so that all but 2 % of the error is the rounding of the result.  A row with an
    infinity or a NaN changes no other; rows of a foreign expert stay as they were."""
    if act_order and (group == -1 or n == WIDE):
        pytest.skip("act-order needs groups; the gather does not depend on the width")
    k, counts = 3200, [64, 3, 250, 0, 40]
    layers = [_layer(k, n, fmt, group, dtype, act_order, dev, seed=i) for i in range(len(counts))]
    emap = torch.tensor([0, 1, 2, 3, -1], dtype=torch.int32, device=dev)
    for foreign in (False, True):
        ids, routing = _routing(counts, dev, emap if foreign else None)
        g = torch.Generator(device=dev).manual_seed(5)
        a = torch.randn(len(ids), k, generator=g, device=dev).to(dtype)
        weights = torch.rand(len(ids), 1, generator=g, device=dev)
        out = _gemm(a, layers[:4] if foreign else layers, routing, n, k, dev, act_order, foreign, weights)
        mine = ids != 4 if foreign else ids >= 0
        ref = torch.zeros(len(ids), n, dtype=torch.float64, device=dev)
        for i, layer in enumerate(layers):
            ref[ids == i] = a[ids == i].double() @ layer[-1]
        ref *= weights.double()
        err = (out.double() - ref)[mine].norm() / (ref.to(dtype).double() - ref)[mine].norm()
        assert float(err) < 1.02
        assert bool((out[~mine] == 7).all())
        b = a.clone()
        b[5, 3], b[17, k - 1] = float("inf"), float("nan")
        other = _gemm(b, layers[:4] if foreign else layers, routing, n, k, dev, act_order, foreign, weights)
        keep = torch.ones(len(ids), dtype=torch.bool, device=dev)
        keep[5] = keep[17] = False
        assert torch.equal(other[keep], out[keep])
        assert not mine[17] or bool(torch.isnan(other[17]).all())


@pytest.mark.parametrize("dtype,fmt", TYPES)
@pytest.mark.parametrize("group,hidden,inter", [(128, 512, 384), (32, 3072, 640), (128, 2944, 7808), (128, 3072, 7808), (-1, 3072, 7808)])
def test_fused_layer_equals_separate_launches(dev, monkeypatch, dtype, fmt, group, hidden, inter):
    """SiLU-and-mul and the sum over experts in the epilogues against separate launches, bit for bit; the last three on wide tiles in GEMM1.  The
    last two cut that GEMM's last tiles along K, others with the epilogue (gate and up columns) than without: fp32 sums in another order, so a few
    intermediate values round the other way, each to a neighbour.  Both layers are sums of thousands of these, so they differ by less than eps in norm."""
    import vllm_amd.fused_marlin_moe as fm
    import vllm_amd.ops as ops
    monkeypatch.setattr(fm, "pick_block_size", lambda *a, **kw: 64)
    e, topk, tokens = 4, 2, 1100 if inter > 4096 else 150
    w = [[_layer(k, n, fmt, group, dtype, False, dev, seed=10 * j + i) for i in range(e)] for j, (k, n) in
         enumerate(((hidden, 2 * inter), (inter, hidden)))]
    (w1, s1, z1), (w2, s2, z2) = ([torch.stack([layer[j] for layer in x]) for j in range(3)] for x in w)
    zeros = dict(w1_zeros=z1, w2_zeros=z2) if fmt == "uint4" else {}
    g = torch.Generator(device=dev).manual_seed(3)
    x = (torch.randn(tokens, hidden, generator=g, device=dev) / hidden ** 0.5).to(dtype)
    logits = torch.randn(tokens, e, generator=g, device=dev)
    weights, ids = torch.softmax(logits, 1).topk(topk, 1)

    def run(**kw):
        return fm.fused_marlin_moe(x, w1, w2, None, None, s1, s2, logits, weights, ids.int(), quant_type_id=w[0][0][5].id, global_num_experts=e, **zeros,
                                   **kw)

    def silu_and_mul(activation, output, input):  # a function of the caller's: separate launches
        fm.default_activation_func(activation, output, input)

    def add(x, out):
        ops.moe_sum(x, out)
        return out

    out = run()
    assert bool(torch.isfinite(out).all()) and float(out.float().norm()) > 0
    separate = run(activation_func=silu_and_mul, moe_sum=add)
    if hidden == 3072 and inter == 7808:
        assert float((out.double() - separate.double()).norm() / separate.double().norm()) < torch.finfo(dtype).eps
    else:
        assert torch.equal(out, separate)
