"""MoE calls past the limits of the kernels that take the others: blocks of 64 with 2 GiB of activations, which gemm_slots.hip does not address
(64-row kernel, gemm_mid.hip), and blocks of 128 in bf16 with uint4b8 weights whose 8-bit terms would exceed their bound (prefill kernel,
gemm_fat.hip).  test_plans.py holds the choice."""
import pytest
import torch

from test_gpu_group_constants import TYPES
from test_gpu_kq_heights import _layer

pytestmark = pytest.mark.gpu

COUNTS = [64, 1, 16, 17, 0, 32, 33, 48, 49, 100]  # tokens of each expert
LARGE_A = [(1 << 20, 1024), (1 << 18, 4096)]      # rows of A and K: 2 GiB; tiles whole and cut along K
LONG_IDS = (4096, 505 * 128)                      # K and slot ids, most of them behind the last live block
N = 192


def _gemm(a, tokens, layers, block, n_ids=None):
    """The rows `tokens` of A, COUNTS of them to each expert; the others belong to none."""
    import vllm_amd.ops as ops
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    from vllm_amd.moe_align_block_size import moe_align_block_size
    dev, m, k = a.device, *a.shape
    mq, ms, mz = (torch.stack([layer[i] for layer in layers]) for i in range(3))
    e = torch.empty((len(layers), 0), dtype=torch.int32, device=dev)
    ids = torch.tensor([x for x, cnt in enumerate(COUNTS) for _ in range(cnt)], dtype=torch.int32, device=dev)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(3)).to(dev)]
    s, x, t = moe_align_block_size(ids[:, None], block, len(layers))
    s = torch.cat([tokens, torch.tensor([m], dtype=torch.int32, device=dev)])[s.long()]
    if n_ids:
        s = torch.cat([s, torch.full((n_ids - len(s),), m, dtype=torch.int32, device=dev)])
        x = torch.cat([x, torch.zeros(n_ids // block - len(x), dtype=torch.int32, device=dev)])
    c = torch.full((m, N), 7.0, dtype=a.dtype, device=dev)
    ops.moe_wna16_marlin_gemm(
        a, c, mq, None, ms, None, mz, e, e, marlin_make_workspace_new(dev, 4), s, x, t, torch.ones(m, 1, device=dev), moe_block_size=block, top_k=1,
        mul_topk_weights=False, is_ep=False, b_q_type=layers[0][5], size_m=m, size_n=N, size_k=k, is_k_full=True, use_atomic_add=False,
        use_fp32_reduce=True, is_zp_float=False)
    out = c[tokens.long()]
    c[tokens.long()] = 7.0
    assert bool((c == 7.0).all())  # rows of no expert stay as they were
    return out, ids


def _check(a, tokens, layers, block, n_ids=None):
    """Rows with a single one pick rows of the weights, bit for bit; random rows to the rounding of the result, 1.66e-3 of the root mean square in bf16
    and an eighth of that in fp16 (test_gpu_kq_heights.py)."""
    dev, k = a.device, a.size(1)
    at = torch.tensor([(r if i % 2 else r + 31) % k for i, r in enumerate(range(0, 32 * len(tokens), 32))], device=dev)
    a[tokens.long(), at] = 1
    out, ids = _gemm(a, tokens, layers, block, n_ids)
    assert torch.equal(out, torch.stack([layers[int(i)][-1][r] for i, r in zip(ids, at)]).to(a.dtype))
    rows = torch.randn(len(tokens), k, generator=torch.Generator(device=dev).manual_seed(2), device=dev).to(a.dtype)
    a[tokens.long()] = rows
    out, _ = _gemm(a, tokens, layers, block, n_ids)
    ref = torch.stack([rows[j].double() @ layers[int(i)][-1] for j, i in enumerate(ids)])
    assert float((out.double() - ref).norm() / ref.norm()) < (1.75e-3 if a.dtype == torch.bfloat16 else 2.3e-4)


@pytest.mark.parametrize("m,k", LARGE_A)
@pytest.mark.parametrize("dtype,fmt", TYPES)
@pytest.mark.parametrize("group", [32, 128, -1])
def test_blocks_of_64(dev, m, k, dtype, fmt, group):
    a = torch.zeros(m, k, dtype=dtype, device=dev)
    tokens = torch.linspace(0, m - 1, sum(COUNTS), dtype=torch.float64).int().to(dev)
    _check(a, tokens, [_layer(k, N, fmt, group, dtype, False, dev, seed=i) for i in range(len(COUNTS))], 64)


@pytest.mark.parametrize("group", [128, 256, -1])
def test_blocks_of_128(dev, group):
    k, n_ids = LONG_IDS
    m = 1000
    a = torch.zeros(m, k, dtype=torch.bfloat16, device=dev)
    tokens = torch.randperm(m, generator=torch.Generator().manual_seed(1))[:sum(COUNTS)].int().to(dev)
    _check(a, tokens, [_layer(k, N, "uint4b8", group, torch.bfloat16, False, dev, seed=i) for i in range(len(COUNTS))], 128, n_ids)
