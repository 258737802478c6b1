"""MoE blocks of 128 slots with bf16 activations and uint4b8 weights on the 8-bit matrix unit (gemm_x8.hip: x8_split_slots_kernel, x8_moe_kernel):
live blocks that are full, partly full and cut along K, fewer columns than a tile, foreign experts, both fused epilogues, act-order, outliers,
infinities and NaNs.  Weights stay exact there, so against the float64 product with unrounded weights an error is what rounding the exact result to
bf16 leaves, r, and the sums' own 0.17 r at most: 1.03 r^2, and the product of the two scatters by 2 * 0.17 / sqrt(192) = 0.025 r^2 over the smallest
result here; three times that is below (1.06 r)^2.  Bound: 1.1 r.  Kernels that round the weights have 1.28 r."""
import pytest
import torch

from test_gpu_x8 import _layer, _rel

pytestmark = pytest.mark.gpu


def _over_rounding(out, ref):
    return float((out.double() - ref).norm() / (ref.bfloat16().double() - ref).norm())


class Moe:
    """E experts [k, n] and a routing of `counts` tokens to each; foreign: expert 1 belongs to another rank."""

    def __init__(self, dev, k, n, counts, group, foreign=False, act_order=False, topk=1):
        from vllm_amd.marlin_utils import marlin_make_workspace_new
        from vllm_amd.moe_align_block_size import moe_align_block_size
        self.k, self.n, self.topk, self.e = k, n, topk, len(counts)
        layers = [_layer(k, n, "uint4b8", group, dev, seed=i, act_order=act_order) for i in range(self.e)]
        self.exact = [layer[4] for layer in layers]
        local = [i for i in range(self.e) if not (foreign and i == 1)]
        self.w, self.s = (torch.stack([layers[i][j] for i in local]) for j in (0, 1))
        none = torch.empty((len(local), 0), dtype=torch.int32, device=dev)
        self.g_idx, self.perm = (torch.stack([layers[i][j] for i in local]) if act_order else none for j in (5, 6))
        ids = torch.tensor([x for x, c in enumerate(counts) for _ in range(c)], dtype=torch.int32, device=dev)
        self.ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(1)).to(dev)].view(-1, topk)
        self.tokens = self.ids.size(0)
        emap = None
        if foreign:
            emap = torch.tensor([0, -1] + list(range(1, self.e - 1)), dtype=torch.int32, device=dev)
        self.weights = torch.rand(self.tokens, topk, generator=torch.Generator(device=dev).manual_seed(2), device=dev)
        self.routing = moe_align_block_size(self.ids, 128, self.e, emap)
        self.workspace, self.foreign = marlin_make_workspace_new(dev, 4), foreign

    def gemm(self, a, mul=True, bias=None):
        import vllm_amd.ops as ops
        from vllm_amd.scalar_type import scalar_types
        s, x, t = self.routing
        c = torch.full((self.tokens * self.topk, self.n), 7.0, dtype=a.dtype, device=a.device)
        return ops.moe_wna16_marlin_gemm(
            a, c, self.w, bias, self.s, None, None, self.g_idx, self.perm, self.workspace, s, x, t, self.weights, moe_block_size=128, top_k=self.topk,
            mul_topk_weights=mul, is_ep=self.foreign, b_q_type=scalar_types.uint4b8, size_m=self.tokens, size_n=self.n, size_k=self.k, is_k_full=True,
            use_atomic_add=False, use_fp32_reduce=True, is_zp_float=False)

    def reference(self, a, mul=True):
        rows = a.double().repeat_interleave(self.topk, 0)
        out, flat = torch.full((len(rows), self.n), 7.0, dtype=torch.float64, device=a.device), self.ids.flatten()
        for i in range(self.e):
            if not (self.foreign and i == 1):
                out[flat == i] = rows[flat == i] @ self.exact[i]
        tw = self.weights.double().flatten()[:, None]
        mine = ~((flat == 1) & self.foreign)
        out[mine] *= tw[mine] if mul else 1
        return out


CASES = [
    # k, n, tokens of each expert, group, foreign, act-order
    (256, 192, [1], 128, False, False),                                 # one live tile
    (4096, 1024, [300, 40, 0, 129, 127, 128], 128, True, False),        # all tiles cut along K
    (2048, 576, [700, 5, 333], 256, False, False),
    (1024, 4160, [128, 1, 260], -1, False, False),                      # last strip one n-tile
    (512, 640, [150, 33], 128, False, True),
    (1024, 16448, [1100, 130, 17, 250], 128, False, False),             # whole tiles in front of cut ones
    (1024, 33344, [300, 1000, 20, 13], -1, False, False),               # more row blocks than a chunk of the tile order
]


def _data(moe, dev, seed=5):
    return torch.randn(moe.tokens, moe.k, generator=torch.Generator(device=dev).manual_seed(seed), device=dev)


@pytest.mark.parametrize("k,n,counts,group,foreign,act_order", CASES)
@pytest.mark.parametrize("mul", [False, True])
def test_against_exact_weights(dev, k, n, counts, group, foreign, act_order, mul):
    moe = Moe(dev, k, n, counts, group, foreign, act_order)
    a = _data(moe, dev).bfloat16()
    out, ref = moe.gemm(a, mul), moe.reference(a, mul)
    assert _over_rounding(out, ref) < 1.1
    if foreign:
        assert bool((out[moe.ids.flatten() == 1] == 7).all())
    assert torch.equal(out, moe.gemm(a, mul))


@pytest.mark.parametrize("k,n,counts,group,foreign,act_order", CASES)
def test_special_values_and_outliers(dev, k, n, counts, group, foreign, act_order):
    """As test_gpu_x8_prepared.py: rows with infinities, NaNs and activations far above the others, and rows without, untouched."""
    moe = Moe(dev, k, n, counts, group, foreign, act_order)
    g = torch.Generator(device=dev).manual_seed(7)
    plain = _data(moe, dev)
    a = plain.clone()
    m = moe.tokens
    rows = torch.arange(0, m, 3, device=dev)
    at = torch.randint(0, k, (len(rows),), generator=g, device=dev)
    a[rows, at] *= 10.0 ** (3 + 6 * torch.rand(len(rows), generator=g, device=dev))
    special = [r for r in (4, m - 1, 40) if r < m]
    for r, (c, v) in zip(special, ((5, float("inf")), (k - 1, float("-inf")), (100, float("nan")))):
        a[r, c] = v
    a, plain = a.bfloat16(), plain.bfloat16()
    out, clean, ref = moe.gemm(a), moe.gemm(plain), moe.reference(a)
    for r in special:
        assert torch.equal(torch.isnan(out[r]), torch.isnan(ref[r]))
        fin = ~torch.isnan(ref[r])
        assert torch.equal(out[r].double()[fin], ref[r][fin].bfloat16().double())
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[rows] = False
    keep[special] = False
    assert torch.equal(out[keep], clean[keep])
    flat = moe.ids.flatten()
    ok = torch.isfinite(ref[rows]).all(1) & ~((flat[rows] == 1) & foreign)
    rows, at = rows[ok], at[ok]
    if len(rows):
        assert _over_rounding(out[rows], ref[rows]) < 1.2  # (beside outliers 0.25 r where their weight is +-1, see test_gpu_x8.py)
        zero = torch.stack([moe.exact[int(flat[r])][c] for r, c in zip(rows, at)]) == 0
        if int(zero.sum()) > 1000:
            assert _over_rounding(out[rows][zero], ref[rows][zero]) < 1.1


@pytest.mark.parametrize("tokens", [200, 1500])
@pytest.mark.parametrize("group", [128, -1])
@pytest.mark.parametrize("special", [False, True])
def test_fused_layer_equals_separate_launches(dev, monkeypatch, tokens, group, special):
    """Both fused epilogues on blocks of 128 against GEMM, silu_and_mul, GEMM and moe_sum, bit for bit, also where rows hold infinities."""
    import vllm_amd.fused_marlin_moe as fm
    from vllm_amd.scalar_type import scalar_types
    monkeypatch.setattr(fm, "pick_block_size", lambda *a, **kw: 128)
    e, hidden, inter, topk = 4, 512, 384, 2
    w = [[_layer(k, n, "uint4b8", group, dev, seed=10 * j + i) for i in range(e)] for j, (k, n) in enumerate(((hidden, 2 * inter), (inter, hidden)))]
    w1, s1, w2, s2 = (torch.stack([layer[j] for layer in x]) for x in w for j in (0, 1))
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(tokens, hidden, generator=g, device=dev)
    if special:
        x[3, 5], x[tokens - 1, 100], x[50, 7] = float("inf"), float("-inf"), float("nan")
        x[::9, 77] *= 1e6
    x = x.bfloat16()
    logits = torch.randn(tokens, e, generator=g, device=dev)
    weights, ids = torch.softmax(logits, 1).topk(topk, 1)
    ids = ids.int()

    def run(**kw):
        return fm.fused_marlin_moe(x, w1, w2, None, None, s1, s2, logits, weights, ids, quant_type_id=scalar_types.uint4b8.id, global_num_experts=e, **kw)

    def silu_and_mul(activation, output, input):  # a function of the caller's: separate launches
        fm.default_activation_func(activation, output, input)

    def add(x, out):
        import vllm_amd.ops as ops
        ops.moe_sum(x, out)
        return out

    fused, separate = run(), run(activation_func=silu_and_mul, moe_sum=add)
    assert torch.equal(torch.isnan(fused), torch.isnan(separate))
    fin = ~torch.isnan(fused)
    assert torch.equal(fused[fin], separate[fin])
    if not special:
        h = torch.zeros(tokens, hidden, dtype=torch.float64, device=dev)
        for t in range(topk):
            for i in range(e):
                rows = ids[:, t] == i
                y = (x[rows].double() @ w[0][i][4]).bfloat16().double()
                y = (torch.nn.functional.silu(y[:, :inter]).bfloat16().double() * y[:, inter:]).bfloat16().double()
                h[rows] += ((y @ w[1][i][4]) * weights[rows, t:t + 1].double()).bfloat16().double()
        assert _rel(fused, h) < 4e-3  # four roundings of 1.66e-3 and less
