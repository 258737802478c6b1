"""The direct eager entries (`linear`, `topk`, `moe` of csrc/torch_ops.cpp) against the operators they stand in for: they take
plain calls and leave to the dispatcher every call that something else has to see, or whose arguments it would convert."""
import numpy as np
import pytest
import torch

from helpers import make_layer
from test_gpu_moe import make_experts, rand_topk

pytestmark = pytest.mark.gpu

M, E, TOPK = 5, 4, 2


class Calls:
    """linear / topk / moe by name, each as a user's program calls it; `value` takes the place of its flag."""

    def __init__(self, dev, monkeypatch):
        from vllm_amd import _custom_ops
        from vllm_amd.marlin_utils import marlin_make_workspace_new
        self.taken = {}  # entry -> whether its last call was answered without the dispatcher
        for name in ("linear", "topk", "moe"):
            entry = getattr(_custom_ops, "eager_" + name)

            def spy(*args, _entry=entry, _name=name):
                out = _entry(*args)
                self.taken[_name] = out is not None
                return out
            monkeypatch.setattr(_custom_ops, "eager_" + name, spy)
        self.layer = make_layer(256, 128, 64, act_order=True)
        self.operands = [t.to(dev) for t in (self.layer.marlin_q, self.layer.marlin_s, self.layer.marlin_zp,
                                             self.layer.g_idx_sorted, self.layer.sort_indices)]
        self.workspace = marlin_make_workspace_new(dev, 4)
        self.experts = [make_experts(E, k, n, 64, torch.float16, False, True, seed=s) for k, n, s in ((256, 512, 1), (256, 256, 2))]
        self.experts = [[t.to(dev) if torch.is_tensor(t) else t for t in o] for o in self.experts]
        g = torch.Generator().manual_seed(3)
        self.x = torch.randn(M, 256, generator=g).half().to(dev)
        self.logits = torch.randn(M, E, generator=g).to(dev)
        self.ids = rand_topk(M, TOPK, E, seed=6).to(dev)
        self.tw = torch.rand(M, TOPK, generator=g).to(dev)

    def linear(self, x=None, value=True, fp32_reduce=True):
        from vllm_amd.marlin_utils import apply_gptq_marlin_linear
        from vllm_amd.scalar_type import scalar_types
        return apply_gptq_marlin_linear(self.x if x is None else x, *self.operands, self.workspace, scalar_types.uint4b8, 128, 256,
                                        value, None, fp32_reduce)

    def topk(self, x=None, value=True, topk=TOPK):
        from vllm_amd.fused_moe import fused_topk
        return fused_topk(self.x, self.logits if x is None else x, topk, value)

    def moe(self, x=None, value=True, is_k_full=True):
        from vllm_amd.fused_marlin_moe import fused_marlin_moe
        (_, q1, s1, _, g1, p1), (_, q2, s2, _, g2, p2) = self.experts
        return fused_marlin_moe(self.x if x is None else x, q1, q2, None, None, s1, s2, None, self.tw, self.ids,
                                quant_type_id=self.layer.type_id, apply_router_weight_on_input=value, global_num_experts=E,
                                g_idx1=g1, g_idx2=g2, sort_indices1=p1, sort_indices2=p2, workspace=self.workspace, is_k_full=is_k_full)

    def input(self, name):
        return self.logits if name == "topk" else self.x


@pytest.fixture
def calls(dev, monkeypatch):
    return Calls(dev, monkeypatch)


def same(a, b):
    a, b = (a, b) if isinstance(a, (tuple, list)) else ((a,), (b,))
    return len(a) == len(b) and all(torch.equal(x.as_subclass(torch.Tensor), y.as_subclass(torch.Tensor))
                                    for x, y in zip(a, b))


NAMES = ["linear", "topk", "moe"]
OPERATOR = {"linear": "gptq_marlin_gemm", "topk": "topk_softmax", "moe": "moe_sum"}


@pytest.mark.parametrize("name", NAMES)
def test_plain_calls_are_taken(calls, name):
    x = calls.input(name)
    getattr(calls, name)()
    assert calls.taken[name]
    for guard in (torch.no_grad, torch.inference_mode):
        with guard():
            getattr(calls, name)(torch.nn.Parameter(x))
            assert calls.taken[name]


# what the dispatcher takes for a bool means the same as that bool, on both sides of the call
@pytest.mark.parametrize("value", [1, 0, np.bool_(True), np.bool_(False), torch.tensor(True), torch.tensor(False)], ids=repr)
@pytest.mark.parametrize("name", NAMES)
def test_flags_that_are_not_bools(calls, name, value):
    call, want = getattr(calls, name), bool(value)
    assert same(call(value=value), call(value=want))
    if name == "linear":
        assert same(call(fp32_reduce=value), call(fp32_reduce=want))
    if name == "moe":
        assert same(call(is_k_full=value), call(is_k_full=want))


def test_counts_that_are_not_ints(calls):
    assert same(calls.topk(topk=np.int64(TOPK)), calls.topk())
    with pytest.raises((TypeError, RuntimeError)):
        calls.topk(topk=2.0)


class Tagged(torch.Tensor):
    seen: list = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(str(func))
        return super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.parametrize("name", NAMES)
def test_tensor_subclass_sees_the_operator(calls, name):
    want = getattr(calls, name)()
    Tagged.seen = []
    got = getattr(calls, name)(calls.input(name).as_subclass(Tagged))
    assert not calls.taken[name] and any(OPERATOR[name] in s or "moe_marlin_gemm_fused" in s for s in Tagged.seen)
    assert same(got, want)
    if name == "linear":
        assert type(got) is Tagged


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("kind", ["function", "dispatch", "profiler"])
def test_modes_see_the_operator(calls, name, kind):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    want, seen = getattr(calls, name)(), []

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    if kind == "profiler":
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            got = getattr(calls, name)()
        seen += [e.key for e in prof.key_averages()]
    else:
        with (Function if kind == "function" else Dispatch)():
            got = getattr(calls, name)()
    assert not calls.taken[name] and any(OPERATOR[name] in s or "moe_marlin_gemm_fused" in s for s in seen), seen
    assert same(got, want)


@pytest.mark.parametrize("name", NAMES)
def test_autograd_goes_through_the_dispatcher(calls, name):
    want = getattr(calls, name)()
    got = getattr(calls, name)(calls.input(name).clone().requires_grad_())
    assert not calls.taken[name]
    assert same([t.detach() for t in got] if name == "topk" else got.detach(), list(want) if name == "topk" else want)


def test_vmap_goes_through_the_dispatcher(calls):
    x = torch.stack([calls.x, calls.x + 1, calls.x * 2])
    want = torch.stack([calls.linear(r) for r in x])
    got = torch.vmap(calls.linear)(x)
    assert not calls.taken["linear"]
    assert torch.equal(got, want)
