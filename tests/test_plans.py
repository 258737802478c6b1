"""Which kernel and tile a call runs on (256 compute units): the GPU tests that list shapes for a tile rely on it, and a changed constant in
the planner must not leave a tile untested."""
import ctypes
import os
import subprocess

import pytest

from vllm_amd import _lib
from vllm_amd import build as vbuild

HERE = os.path.dirname(os.path.abspath(__file__))
FIELDS = ["kind", "mb", "tn", "splits", "kps", "ks", "tail_strips", "tail_kind", "tail_mb", "xcd_map",
          "scratch_kib", "first_scratch_kib", "first_kind"]


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    import torch
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("no hipcc")
    if torch.cuda.is_available():
        pytest.skip("the planner asks the GPU for its compute units")
    _lib.load()
    out = str(tmp_path_factory.mktemp("plan") / "plan_probe.so")
    libdir = os.path.dirname(vbuild.LIB_PATH)
    subprocess.run([vbuild.hipcc_path()] + vbuild.HIPCC_FLAGS + ["-O1", os.path.join(HERE, "plan_probe.hip"), "-o", out, f"-L{libdir}",
                                                                  f"-l:{vbuild.LIB_NAME}", f"-Wl,-rpath,{libdir}"],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    probe = ctypes.CDLL(out).plan_probe

    def call(m, k, n, dtype, fmt, group, act_order=False, more_scratch=True, moe_slots=0, moe_block=64):
        """`dtype`: a torch dtype; operands are never read.  moe_slots: MoE blocks of `moe_block` and so many sorted slots."""
        a = _lib.GemmArgs()
        a.struct_size = ctypes.sizeof(_lib.GemmArgs)
        a.dtype = _lib.DTYPE_BF16 if dtype == torch.bfloat16 else _lib.DTYPE_F16
        a.wtype = _lib.WTYPE_U4B8 if fmt == "uint4b8" else _lib.WTYPE_U4
        a.flags = _lib.F_IS_K_FULL | _lib.F_USE_FP32_REDUCE
        a.a = a.c = a.b_q_weight = a.b_scales = a.workspace = 4096
        a.lda = k + 64
        if fmt == "uint4":
            a.b_zeros = 4096
        if act_order:
            a.g_idx = a.perm = 4096
        a.size_m, a.size_n, a.size_k, a.num_groups = m, n, k, 1 if group == -1 else k // group
        if moe_slots:
            a.flags |= _lib.F_MOE
            a.lda, a.moe_block_size, a.top_k, a.n_sorted = k, moe_block, 1, moe_slots
            a.sorted_token_ids = a.expert_ids = a.num_tokens_past_padded = 4096
        a.workspace_len = 1024  # what marlin_make_workspace_new makes on this GPU
        res = (ctypes.c_int32 * len(FIELDS))()
        assert probe(ctypes.byref(a), int(more_scratch), res) == 0
        return dict(zip(FIELDS, res))

    return call


def test_runs_of_tiles_for_an_xcd(plan):
    """K-split tiles in runs where the L2s share weight strips, and not where the tiles of an XCD share rows (or nothing)."""
    import torch
    f16 = torch.float16
    for m, k, n, act, tile, runs in [
            (203, 4096, 4096, False, (2, 128), 1),
            (37, 4096, 28672, False, (3, 128), 0),    # one row tile
            (512, 4096, 4096, True, (4, 128), 0),     # eight of them behind the gather
            (512, 4096, 6144, True, (4, 256), 0),
            (640, 4096, 6144, False, (4, 256), 1),    # ten
            (300, 14336, 4096, True, (5, 256), 1),    # four, K splits
            (3000, 14336, 4096, False, (6, 256), 0)]:
        p = plan(m, k, n, f16, "uint4b8", 128, act)
        assert (p["kind"], p["mb"], p["tn"], p["xcd_map"]) == (5,) + tile + (runs,), (m, k, n, p)


def test_shapes_of_the_8_bit_unit(plan):
    """Every shape of test_gpu_x8.py runs on the tile it is listed with, whatever the weights, and on the 16-bit kernels without scratch."""
    import test_gpu_x8 as x8
    import torch
    for (k, n, m), tile in x8.SHAPES.items():
        for fmt, group, act in [w + (False,) for w in x8.WEIGHTS] + [("uint4b8", 128, True)]:
            if group < 0 or k % group == 0:
                p = plan(m, k, n, torch.bfloat16, fmt, group, act)
                assert (p["kind"], p["ks"], p["mb"], p["tn"], p["splits"]) == (6,) + tile, (k, n, m, fmt, group, act, p)
    for k, n, m in x8.ENTRY:
        assert plan(m, k, n, torch.bfloat16, "uint4b8", 128)["kind"] == 6
        assert plan(m, k, n, torch.bfloat16, "uint4b8", 128, more_scratch=False)["kind"] != 6
    assert {t[:3] for t in x8.SHAPES.values()} == {(1, 8, 512), (1, 8, 256), (2, 8, 256), (2, 7, 256), (2, 6, 256), (2, 5, 256)}


def test_cold_weights_decide(plan):
    """Plans that times on cached weights got wrong (microseconds on rotated ones): the 8-bit unit for zero points at many rows (2048 x 4096 x
    28672: 432 against 417; 4096 x 8192 x 10240: 602 against 570) and where it saves nothing."""
    import torch
    for m, k, n, fmt, group in [(2048, 4096, 28672, "uint4", 128), (4096, 8192, 10240, "uint4", 128), (4096, 8192, 8192, "uint4", 128),
                                (384, 4096, 6144, "uint4", -1), (384, 4096, 6144, "uint4", 128)]:
        assert plan(m, k, n, torch.bfloat16, fmt, group)["kind"] != 6, (m, k, n)
    for m, k, n in [(512, 4096, 28672), (1024, 8192, 10240), (4096, 4096, 28672)]:
        assert plan(m, k, n, torch.bfloat16, "uint4b8", 128)["kind"] == 6, (m, k, n)


def test_shapes_of_the_k_split_tiles(plan):
    """Every pinned shape of test_gpu_kq_heights.py runs on its tile; together they run every tile in both types, the private K parts' forms that few
    problems reach, and every second pass."""
    import test_gpu_kq_heights as kq
    import torch
    kernels, second_passes = set(), set()
    for (dtype, fmt, group, act), shapes in kq.PINNED.items():
        for (m, k, n), (mb, tn, splits) in shapes.items():
            p = plan(m, k, n, dtype, fmt, group, act)
            if tn:
                got = (p["kind"], p["mb"], p["tn"], p["splits"])
            else:
                got = (p["kind"] + 3 if p["tail_strips"] and p["tail_kind"] == 5 else -1, p["tail_mb"], 0, 1)
            assert got == (5, mb, tn, splits), (m, k, n, dtype, fmt, group, act, p)
            bf16, channel = dtype == torch.bfloat16, group == -1
            kernels.add((mb, tn, bf16) + ((fmt, "column" if channel else "short" if group < 128 else "long") if tn == 128 else ()))
            if splits > 1:
                second_passes.add((tn, bf16, channel))
    assert {(mb, 256, bf16) for mb in (5, 6, 7, 8) for bf16 in (False, True)} <= kernels
    assert {(2, 128, False), (2, 128, True)} <= {x[:3] for x in kernels}
    assert {(mb, 128, True, "uint4", "short") for mb in (2, 3)} <= kernels
    assert {(tn, bf16, channel) for tn in (128, 256) for bf16 in (False, True) for channel in (False, True)} <= second_passes
    assert any(m <= 128 and tn == 256 for s in kq.PINNED.values() for (m, _, _), (_, tn, _) in s.items())


def test_64_row_kernel_of_the_constants_test(plan):
    import test_gpu_group_constants as gc
    for dtype, fmt in gc.TYPES:
        for group in (32, 64, 128, 256, -1):
            assert plan(*gc.DENSE, dtype, fmt, group)["kind"] == 3


def test_prepared_weights(plan):
    """The pinned shapes of test_gpu_x8_prepared.py have their weights prepared; without room for them they run on other kernels."""
    import test_gpu_x8_prepared as xp
    import torch
    for (k, n, m), group in [(s, g) for g, s in xp.WEIGHTS if s in xp.PINNED] + [(xp.OVER_STATIC, 128)]:
        p = plan(m, k, n, torch.bfloat16, "uint4", group)
        assert (p["kind"], p["ks"], p["mb"], p["tn"], p["splits"]) == (7, 1, 8, 512, 1), (k, n, m, group, p)
        assert plan(m, k, n, torch.bfloat16, "uint4", group, more_scratch=False)["kind"] != 7
        assert plan(m, k, n, torch.float16, "uint4", group)["kind"] != 7


def test_moe_blocks_of_64(plan):
    """256-column tiles until 512-column ones number 9/4 (fp16) or 3 (bf16) of the compute units; operands of 2 GiB and more run on the 64-row kernel."""
    import torch
    for dtype in (torch.float16, torch.bfloat16):
        for fmt in ("uint4", "uint4b8"):
            for group in (32, 128, -1):
                blocks = 72 if dtype == torch.float16 else 96      # 8 strips to a block
                for slots, k, n, kind, tn in [
                        (64, 128, 64, 8, 256),
                        (64 * (blocks - 1), 2048, 4096, 8, 256),
                        (64 * (blocks - 1) + 1, 2048, 4096, 8, 512),
                        (64 * 96, 4096, 3648, 8, 512),
                        (64 * 8, 65536, 65536 - 64, 8, 512),       # an expert just under 2 GiB of weights
                        (64 * 8, 65536, 65536, 3, 512)]:
                    got = plan(min(slots, 4096), k, n, dtype, fmt, group, moe_slots=slots)
                    assert (got["kind"], got["tn"], got["splits"]) == (kind, tn, 1), (slots, k, n, group, got)
    rows = (1 << 31) // (2 * 4096)
    assert plan(rows - 1, 4096, 512, torch.bfloat16, "uint4", 128, moe_slots=rows)["kind"] == 8
    assert plan(rows, 4096, 512, torch.bfloat16, "uint4", 128, moe_slots=rows)["kind"] == 3
    # act-order: the gathered rows, one for each slot, are what the kernel reads
    assert plan(rows - 1, 4096, 512, torch.bfloat16, "uint4b8", 128, act_order=True, moe_slots=rows)["kind"] == 3


def test_extra_scratch_has_a_bound(plan):
    """Prepared weights and the terms of MoE rows take 512 MiB at most; problems beyond that run without them."""
    import torch
    assert plan(4096, 8192, 65536, torch.bfloat16, "uint4", 128)["kind"] == 7
    assert plan(4096, 8192, 65536 + 64, torch.bfloat16, "uint4", 128)["kind"] != 7
    slots = 504 * 128                       # rows of 4096 x 2 bytes and 32 scale words
    assert plan(4096, 4096, 2048, torch.bfloat16, "uint4b8", 128, moe_slots=slots, moe_block=128)["kind"] == 9
    assert plan(4096, 4096, 2048, torch.bfloat16, "uint4b8", 128, moe_slots=slots + 1, moe_block=128)["kind"] == 2
    assert plan(4096, 4096, 2048, torch.bfloat16, "uint4b8", 128, more_scratch=False, moe_slots=8192, moe_block=128)["kind"] == 2


def test_moe_blocks_of_128(plan):
    """bf16 uint4b8 with groups of whole 128 rows or one scale per column runs on the 8-bit unit, everything else on the prefill kernel."""
    import torch
    for dtype in (torch.float16, torch.bfloat16):
        for fmt in ("uint4", "uint4b8"):
            for group in (32, 64, 128, 256, -1):
                for slots, k, n in [(128, 256, 64), (9208, 4096, 28672), (9208, 14336, 4096)]:
                    x8 = dtype == torch.bfloat16 and fmt == "uint4b8" and group not in (32, 64)
                    assert plan(128, k, n, dtype, fmt, group, moe_slots=slots, moe_block=128)["kind"] == (9 if x8 else 2), (dtype, fmt, group, k)
    assert plan(128, 4096, 4096, torch.bfloat16, "uint4b8", 128, act_order=True, moe_slots=9208, moe_block=128)["kind"] == 9
    assert plan(128, 65536, 65536 - 64, torch.bfloat16, "uint4b8", 128, moe_slots=128, moe_block=128)["kind"] == 9
    assert plan(128, 65536, 65536, torch.bfloat16, "uint4b8", 128, moe_slots=128, moe_block=128)["kind"] == 2  # 2 GiB of an expert's weights


def test_moe_beyond_limits(plan):
    """The calls of test_gpu_moe_beyond_limits.py."""
    import test_gpu_moe_beyond_limits as bl
    import torch
    for dtype, fmt in bl.TYPES:
        for group in (32, 128, -1):
            for m, k in bl.LARGE_A:
                assert plan(m, k, bl.N, dtype, fmt, group, moe_slots=990)["kind"] == 3
    k, ids = bl.LONG_IDS
    for group in (128, 256, -1):
        assert plan(1000, k, bl.N, torch.bfloat16, "uint4b8", group, moe_slots=ids, moe_block=128)["kind"] == 2
        assert plan(1000, k, bl.N, torch.bfloat16, "uint4b8", group, moe_slots=ids - 128, moe_block=128)["kind"] == 9


def test_tiles_of_rows_with_unscaled_weights(plan):
    """The shapes of test_gpu_rows.py run on the tile they are listed with; what the kernel does not take, and what has never run on 16-row tiles, stays."""
    import torch
    import test_gpu_rows as rows
    tiles, uneven, splits = set(), set(), set()
    for (m, k, n, dtype, fmt, group, act), (mb, sp, units) in rows.ROWS.items():
        p = plan(m, k, n, dtype, fmt, group, act)
        assert (p["kind"], p["mb"], p["splits"], p["kps"], p["tn"]) == (10, mb, sp, 4 * units, 64), (m, k, n, dtype, fmt, group, p)
        tiles.add((mb, dtype, fmt, group == -1))
        splits.add((mb, sp))
        if k // 128 % units:
            uneven.add((mb, sp))
        # no more scratch than the 16-row tiles take, where a caller asks for little: with this many splits those keep the problem
        less = plan(m, k, n, dtype, fmt, group, act, more_scratch=False)
        assert less["first_kind"] == 1 and less["scratch_kib"] <= less["first_scratch_kib"], (m, k, n, less)
        assert less["kind"] == (1 if sp > 1 else 10) and (sp == 1 or p["scratch_kib"] > p["first_scratch_kib"]), (m, k, n, less)
        assert plan(16, k, n, dtype, fmt, group, act)["kind"] == 1 and plan(49, k, n, dtype, fmt, group, act)["kind"] != 10
    for m, k, n, group in [(37, 14336, 4096, 64), (37, 14336 + 64, 4096, -1), (37, 14336, 4096, 32), (37, 4096, 4096, 128), (37, 4096, 28672, 128),
                           (20, 4096, 64 * 257, 128)]:
        assert plan(m, k, n, torch.bfloat16, "uint4", group)["kind"] != 10, (m, k, n, group)
    assert {(mb, s) for mb in (2, 3) for s in (2, 5, 7)} <= uneven and {(3, 1), (2, 4), (3, 3), (3, 4)} <= splits
    assert {t[:3] for t in tiles} >= {(3, dt, fmt) for dt in (torch.float16, torch.bfloat16) for fmt in ("uint4", "uint4b8")}


def test_static_and_repeated_calls_on_tiles_of_rows(plan):
    """The calls of test_zz_no_alloc.py and test_gpu_splitk_stress.py that stand for the exchange between K splits of 32- and 48-row tiles."""
    import test_gpu_splitk_stress as stress
    import test_zz_no_alloc as static
    import torch
    k, n, group, dtype, zp, act, ms = static.ROWS_CASE
    assert [(p["kind"], p["mb"], p["splits"]) for p in (plan(m, k, n, dtype, "uint4" if zp else "uint4b8", group, act) for m in ms)] == [(10, 3, 4), (10, 2, 4)]
    got = [plan(m, k, n, torch.float16, "uint4b8", 128) for _, m, k, n in stress.ROWS_CASES]
    assert [(p["kind"], p["mb"], p["splits"]) for p in got] == [(10, 3, 4), (10, 2, 4)]
