"""64-row tiles (dense: gemm_mid.hip; MoE: gemm_slots.hip, and gemm_mid.hip in test_gpu_moe_beyond_limits.py): dequantisation constants made once per 128 rows of K (groups of 128 rows and more, one scale per column) and with
every k-step (shorter groups).  A row of A with a single one picks one row of the weights: the result is that row, bit for bit, for every
group boundary, word position and half of a column tile."""
import pytest
import torch

from test_gpu_kq_heights import _layer, _run

pytestmark = pytest.mark.gpu

TYPES = [(torch.float16, "uint4b8"), (torch.float16, "uint4"), (torch.bfloat16, "uint4b8"), (torch.bfloat16, "uint4")]
DENSE = (130, 512, 32832)  # a 64-column last strip; held to the 64-row kernel by test_plans.py


def _one_hot(m, k, dtype, dev):
    """m rows with a one each: both sides of every boundary of 32 K rows, then anywhere."""
    at = [r for b in range(0, k, 32) for r in (b, b + 31)]
    at = (at + [(37 * i) % k for i in range(m)])[:m]
    rows = torch.tensor(at, device=dev)
    a = torch.zeros(m, k, dtype=dtype, device=dev)
    a[torch.arange(m, device=dev), rows] = 1
    return a, rows


@pytest.mark.parametrize("dtype,fmt", TYPES)
@pytest.mark.parametrize("group", [32, 64, 128, 256, -1])
def test_dense_one_hot_rows(dev, dtype, fmt, group):
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    m, k, n = DENSE
    layer = _layer(k, n, fmt, group, dtype, False, dev)
    a, rows = _one_hot(m, k, dtype, dev)
    assert torch.equal(_run(a, layer, n, k, marlin_make_workspace_new(dev)), layer[-1][rows].to(dtype))


@pytest.mark.parametrize("dtype,fmt", TYPES)
@pytest.mark.parametrize("group", [32, 64, 128, 256, -1])
def test_moe_one_hot_rows(dev, dtype, fmt, group):
    """Blocks of 64 slots that hold 1 .. 64 rows, fewer columns than a tile has."""
    import vllm_amd.ops as ops
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    from vllm_amd.moe_align_block_size import moe_align_block_size
    k, n = 512, 192
    counts = [64, 1, 16, 17, 0, 32, 33, 48, 49, 100]  # tokens of each expert
    layers = [_layer(k, n, fmt, group, dtype, False, dev, seed=i) for i in range(len(counts))]
    mq, ms, mz = (torch.stack([layer[i] for layer in layers]) for i in range(3))
    e = torch.empty((len(counts), 0), dtype=torch.int32, device=dev)
    ids = torch.tensor([x for x, cnt in enumerate(counts) for _ in range(cnt)], dtype=torch.int32, device=dev)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(3)).to(dev)]
    a, rows = _one_hot(len(ids), k, dtype, dev)
    s, x, t = moe_align_block_size(ids[:, None], 64, len(counts))
    out = ops.moe_wna16_marlin_gemm(
        a, None, mq, None, ms, None, mz, e, e, marlin_make_workspace_new(dev, 4), s, x, t, torch.ones(len(ids), 1, device=dev), moe_block_size=64,
        top_k=1, mul_topk_weights=False, is_ep=False, b_q_type=layers[0][5], size_m=len(ids), size_n=n, size_k=k, is_k_full=True,
        use_atomic_add=False, use_fp32_reduce=True, is_zp_float=False)
    want = torch.stack([layers[int(i)][-1][r] for i, r in zip(ids, rows)]).to(dtype)
    assert torch.equal(out, want)
