"""Dense bf16 problems of more than 128 rows on the 8-bit matrix unit (gemm_x8.hip): every tile shape, remainders of rows, columns and
K steps, K splits, zero points, groups of 128 and 256 rows and channel-wise scales.

The weights stay exact there (their scale is applied to the fp32 sum), so results are held to the float64 product with the unrounded
weights (q - z) * s.  What is left is the bf16 rounding of the result: its error is at most 2^-9 of a value, 2^-8 / sqrt(12) = 1.13e-3
of it at the bottom of a binade and half of that at the top, and 1.66e-3 of the root mean square on the bell-shaped results here.  The
activations' two 8-bit terms and the unit's 8-element sums add 2e-5 of that.  Bound: 1.75e-3; the kernels that round the weights to bf16 reach
2.1e-3 and more, so the bound also shows which kernel ran."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (K, N, M): tile shapes and splits they run on
SHAPES = [
    (1024, 16448, 512),   # 128 x 512 tiles, last strip one n-tile
    (1152, 8256, 203),    # 128 x 256 tiles of four wavefronts, nine K steps split three ways across workgroups
    (1664, 16448, 350),   # the same unsplit with zero points; two K parts of seven and six steps without
    (2944, 16448, 384),   # two K parts of twelve and eleven steps, 128 rows
    (4096, 16448, 300),   # ... 112 rows
    (3328, 16448, 250),   # ... 96 rows
    (2944, 16448, 190),   # ... 80 rows
]
WEIGHTS = [("uint4b8", 128), ("uint4", 128), ("uint4", -1), ("uint4b8", -1), ("uint4", 256)]


@pytest.fixture
def workspace(dev):
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    return marlin_make_workspace_new(dev)


def _layer(k, n, fmt, group, dev, seed=0):
    """Marlin operands and the unrounded weights in float64."""
    from vllm_amd.marlin_utils import marlin_permute_scales, marlin_zero_points
    from vllm_amd.marlin_utils_test import quantize_weights
    from vllm_amd.quant_utils import gptq_pack
    from vllm_amd.scalar_type import scalar_types as st
    import vllm_amd.ops as ops
    g = torch.Generator(device=dev).manual_seed(seed)
    w = (torch.randn(k, n, generator=g, device=dev) * 0.02).bfloat16()
    wtype, gs = (st.uint4, st.uint4b8)[fmt == "uint4b8"], k if group == -1 else group
    _, q, s, z = quantize_weights(w, wtype, gs, zero_points=fmt == "uint4", rule="absmax")
    e = torch.empty(0, dtype=torch.int32, device=dev)
    exact = ((q.view(k // gs, gs, n).double() - (8 if z is None else z.view(-1, 1, n).double())) * s.view(-1, 1, n).double()).view(k, n)
    mq = ops.gptq_marlin_repack(gptq_pack(q, 4, k, n), e, k, n, 4)
    mz = e if z is None else marlin_zero_points(z, k // gs, n, 4)
    return mq, marlin_permute_scales(s, k, n, gs), mz, wtype, exact


def _run(a, layer, n, k, workspace, bias=None):
    import vllm_amd.ops as ops
    mq, ms, mz, wtype, _ = layer
    e = torch.empty(0, dtype=torch.int32, device=a.device)
    return ops.gptq_marlin_gemm(a, None, mq, bias, ms, None, mz, e, e, workspace, wtype, a.shape[0], n, k, True, False, True, False)


def _rel(out, ref):
    return float((out.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("k,n,m,fmt,group", [s + w for s in SHAPES for w in WEIGHTS if w[1] < 0 or s[0] % w[1] == 0])
def test_against_exact_weights(dev, workspace, k, n, m, fmt, group):
    print(f"x8 k={k} n={n} m={m} {fmt} group={group}", flush=True)
    from vllm_amd.marlin_utils import marlin_permute_bias
    layer = _layer(k, n, fmt, group, dev)
    g = torch.Generator(device=dev).manual_seed(m)
    wide = torch.randn(m, k + 64, generator=g, device=dev).bfloat16()
    a = wide[:, 32:32 + k]  # a strided view
    ref = a.double() @ layer[4]
    out = _run(a, layer, n, k, workspace)
    assert _rel(out, ref) < 1.75e-3
    assert torch.equal(out, _run(a.contiguous(), layer, n, k, workspace))
    bias = torch.randn(n, generator=g, device=dev).bfloat16()
    assert _rel(_run(a, layer, n, k, workspace, marlin_permute_bias(bias)), ref + bias.double()) < 1.75e-3
    assert int(workspace.abs().sum()) == 0


@pytest.mark.parametrize("k,n,m", [SHAPES[0], SHAPES[2], SHAPES[3]])
@pytest.mark.parametrize("fmt,group", [("uint4b8", 128), ("uint4", 128), ("uint4", -1)])
def test_one_hot_rows(dev, workspace, k, n, m, fmt, group):
    """Rows +-2^e * (unit vector), e from one end of bf16's exponents to the other: single products, exact to the last bit."""
    layer = _layer(k, n, fmt, group, dev, seed=1)
    r = torch.arange(m, device=dev)
    ks, e = (7 * r) % k, (r % 220) - 120
    a = torch.zeros(m, k, device=dev, dtype=torch.bfloat16)
    a[r, ks] = torch.where(r % 2 == 0, 1.0, -1.0).to(dev).mul(torch.ldexp(torch.ones(m, device=dev, dtype=torch.float64), e)).bfloat16()
    ref = a[r, ks].double().unsqueeze(1) * layer[4][ks]
    normal = ref.abs() >= 2.0 ** -118  # (below: fp32 and bf16 subnormals on the way)
    out = _run(a, layer, n, k, workspace)
    assert torch.equal(torch.where(normal, out.double(), 0), torch.where(normal, ref.bfloat16().double(), 0))


@pytest.mark.parametrize("kind", ["outliers", "wide", "positive", "offset", "subnormal_rows"])
@pytest.mark.parametrize("k,n,m", [(4096, 16448, 300), (1152, 8256, 203)])
@pytest.mark.parametrize("fmt", ["uint4b8", "uint4"])
def test_activation_distributions(dev, workspace, kind, k, n, m, fmt):
    """Activations that strain the two 8-bit terms (14 binades at full precision below a step's largest value, 22 bits in all) and the
    offset taken out of the sums.  Bound: what a kernel that rounds the weights to bf16 has, 2.5e-3."""
    layer = _layer(k, n, fmt, 128, dev, seed=2)
    g = torch.Generator(device=dev).manual_seed(5)
    a = torch.randn(m, k, generator=g, device=dev)
    if kind == "outliers":
        a[:, 17::128] *= 1000
    elif kind == "wide":
        a *= torch.exp(2 * torch.randn(m, k, generator=g, device=dev))
    elif kind == "positive":
        a = a.abs() + 0.5
    elif kind == "offset":
        a += 8
    else:
        a[::3] *= 2.0 ** -110
        a[5] = 0
    a = a.bfloat16()
    ref = a.double() @ layer[4]
    out = _run(a, layer, n, k, workspace)
    rows = (out.double() - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-300)
    assert float(rows.max()) < 2.5e-3


@pytest.mark.parametrize("k,n,m", [SHAPES[0], SHAPES[2], SHAPES[3]])
@pytest.mark.parametrize("fmt,group", [("uint4b8", 128), ("uint4", 128), ("uint4", -1)])
def test_infinities_and_nans(dev, workspace, k, n, m, fmt, group):
    """A row with infinities or NaNs gives what the float64 product gives (inf, -inf, NaN for inf * 0 and inf - inf); other rows are
    untouched."""
    layer = _layer(k, n, fmt, group, dev, seed=3)
    a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(7), device=dev).bfloat16()
    clean = _run(a, layer, n, k, workspace)
    b = a.clone()
    b[3, 5] = float("inf")
    b[17, k - 1] = float("-inf")
    b[40, 100] = float("nan")
    b[m - 1, 0], b[m - 1, k // 2 + 1] = float("inf"), float("inf")
    rows = [3, 17, 40, m - 1]
    out, ref = _run(b, layer, n, k, workspace), b[rows].double() @ layer[4]
    assert torch.equal(torch.isnan(out[rows]), torch.isnan(ref))
    fin = ~torch.isnan(ref)
    assert torch.equal(out[rows].double()[fin], ref[fin])
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[rows] = False
    assert torch.equal(out[keep], clean[keep])


def _c_args(lib_mod, a, c, layer, n, k, groups):
    args = lib_mod.GemmArgs()
    args.struct_size = ctypes.sizeof(lib_mod.GemmArgs)
    args.dtype, args.wtype, args.flags = lib_mod.DTYPE_BF16, lib_mod.WTYPE_U4B8, lib_mod.F_IS_K_FULL | lib_mod.F_USE_FP32_REDUCE
    args.a, args.lda, args.c = a.data_ptr(), a.stride(0), c.data_ptr()
    args.b_q_weight, args.b_scales = layer[0].data_ptr(), layer[1].data_ptr()
    args.size_m, args.size_n, args.size_k, args.num_groups = a.shape[0], n, k, groups
    return args


@pytest.mark.parametrize("k,n,m", [(1024, 16448, 512), (8192, 2048, 4224)])
def test_entry_points_without_room_for_the_terms(dev, k, n, m):
    """The C entry point with no scratch, and the static one when the split activations exceed its buffer, take the 16-bit kernels
    (whose error is above the 8-bit unit's bound)."""
    from vllm_amd import _lib
    lib = _lib.load()
    layer = _layer(k, n, "uint4b8", 128, dev, seed=4)
    a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(9), device=dev).bfloat16()
    ref = a.double() @ layer[4]
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    ws = torch.zeros(4096, dtype=torch.int32, device=dev)

    def call(fn, scratch):
        c = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
        args = _c_args(_lib, a, c, layer, n, k, k // 128)
        args.workspace, args.workspace_len = ws.data_ptr(), ws.numel()
        need = lib.w4a16_gemm_scratch_bytes(ctypes.byref(args))
        buf = torch.empty(max(need, 4), dtype=torch.uint8, device=dev) if scratch else None
        args.c_tmp = buf.data_ptr() if scratch else None
        assert fn(ctypes.byref(args), stream) == 0, lib.w4a16_last_error()
        torch.cuda.synchronize()
        return _rel(c, ref), need

    err, need = call(lib.w4a16_marlin_gemm, True)
    assert err < 1.75e-3 and need > 2 * m * k
    assert 1.75e-3 < call(lib.w4a16_marlin_gemm, False)[0] < 2.5e-3
    err = call(lib.w4a16_marlin_gemm_static, False)[0]
    assert err < 1.75e-3 if need <= _lib.STATIC_SCRATCH_BYTES else 1.75e-3 < err < 2.5e-3
