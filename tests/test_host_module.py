"""The C++ host module's entry points where no kernel runs: what they refuse, and how they find the weights."""
import pytest
import torch
import torch.nn.utils.parametrize
import torch.autograd.forward_ad as fwAD

from optimus import _native as _n

T, H, I, N, K = 4, 16, 8, 3, 2


def _tensors():
    g = torch.Generator().manual_seed(0)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    i32 = lambda n: torch.zeros(n, dtype=torch.int32)
    return dict(x=rnd(T, H), weight=rnd(N, H), bias=torch.zeros(N), rw=rnd(T, K), residual=rnd(T, H), y=rnd(T * K, H),
                gate=rnd(N, I, H), up=rnd(N, I, H), down=rnd(N, H, I),
                experts=torch.zeros(T, K, dtype=torch.int64), cum=i32(N + 1), cum_ep=i32(T + 1), rows=i32(T * K))


def _calls():
    """entry point -> (call on a dict of tensors, the names of its differentiable inputs)"""
    h = _n.host()
    leaves = lambda t: [t["gate"], t["up"], t["down"]]
    return {
        "gate_logits": (lambda t: h.gate_logits(t["x"], t["weight"]), ("x", "weight")),
        "route_softmax": (lambda t: h.route_softmax(t["x"], t["weight"], K, False, torch.bfloat16, False, False),
                          ("x", "weight")),
        "route_sigmoid": (lambda t: h.route_sigmoid(t["x"], t["weight"], t["bias"], 1, 1, K, True, 1.0),
                          ("x", "weight", "bias")),
        "moe_experts": (lambda t: h.moe_experts(t["x"], t["rw"], t["experts"], 0, N, N, False, t["residual"], True,
                                                leaves(t), False, None),
                        ("x", "rw", "residual", "gate", "up", "down")),
        "merged_mlp": (lambda t: h.merged_mlp(t["x"], t["cum"], True, leaves(t), None, None, None),
                       ("x", "gate", "up", "down")),
        "combine": (lambda t: h.combine(t["y"], t["rw"], t["cum_ep"], t["rows"], t["rows"], t["rows"], t["residual"]),
                    ("y", "rw", "residual")),
    }


CASES = [("gate_logits", 2), ("route_softmax", 2), ("route_sigmoid", 3), ("moe_experts", 6), ("merged_mlp", 4),
         ("combine", 3)]


@pytest.mark.parametrize("name,at", [(name, at) for name, n in CASES for at in range(n)])
def test_forward_mode_is_refused(name, at):
    """A tangent on any differentiable input raises what an autograd function without a jvp raises; it used to be
    dropped without a word."""
    call, inputs = _calls()[name]
    assert len(inputs) == dict(CASES)[name]
    t = _tensors()
    with fwAD.dual_level():
        t[inputs[at]] = fwAD.make_dual(t[inputs[at]], torch.ones_like(t[inputs[at]]))
        with pytest.raises(NotImplementedError, match="jvp"):
            call(t)


@pytest.mark.parametrize("name", [name for name, _ in CASES])
@pytest.mark.parametrize("transform", [torch.vmap, torch.func.grad])
def test_functorch_transforms_are_refused(name, transform):
    call, inputs = _calls()[name]
    t = _tensors()
    first = torch.stack([t[inputs[0]]] * 2) if transform is torch.vmap else t[inputs[0]]

    def f(v):
        call({**t, inputs[0]: v})
        return v.sum()
    with pytest.raises(RuntimeError, match="torch.func transforms|jvp"):
        transform(f)(first)


def test_block_finds_a_parametrized_merged_weight():
    """(on the CPU the fused path declines the operands, which it does after it has found the weights)"""
    from optimus.mapper import ParallelDpPpEpTpMapper
    from optimus.models.common.moe import FastOlmoeParallelSparseMoeBlock
    from optimus.models.olmoe.configuration_olmoe import OlmoeParallelConfig
    cfg = OlmoeParallelConfig(hidden_size=H, intermediate_size=I, num_experts=N, num_experts_per_tok=K, use_fast_moe=True,
                              use_merged_mlp_in_fast_moe=True)
    blk = FastOlmoeParallelSparseMoeBlock(cfg, ParallelDpPpEpTpMapper())
    torch.nn.utils.parametrize.register_parametrization(blk.experts, "gate_proj_merged_weight", torch.nn.Identity())
    t = _tensors()
    assert blk._fused_experts_fn(t["x"].float(), t["rw"], t["experts"], None) is None


def test_the_functions_are_autograd_functions():
    """Callers subclass them, and call their forward and backward."""
    from optimus.models.common import moe
    for name in ("GateLogitsFunction", "GateLogitsF32Function", "GateSoftmaxTopkFunction", "SoftmaxTopkRouterFunction",
                 "GroupedGemmFunction", "MergedMLPFunction", "GatheredMergedMLPFunction", "GroupMLPFunction",
                 "GatheredGroupMLPFunction", "RoutedMLPFunction", "RoutedAndSharedMLPFunction",
                 "PrepareInputForGroupGemmFunction", "GroupGemmOutputReductionFunction",
                 "GroupGemmOutputReductionResidualFunction"):
        cls = getattr(moe, name)
        assert issubclass(cls, torch.autograd.Function), name
        assert "forward" in vars(cls) and "backward" in vars(cls), name


@pytest.mark.parametrize("name,changes", [
    ("gate_logits", dict(x=lambda t: t.float())), ("gate_logits", dict(weight=lambda t: t.float())),
    ("gate_logits", dict(weight=lambda t: t[:, :8])), ("gate_logits", dict(x=lambda t: t[0])),
    ("route_softmax", dict(x=lambda t: t.float())), ("route_softmax", dict(weight=lambda t: t[:, :8].contiguous())),
    ("route_sigmoid", dict(weight=lambda t: t.float())), ("route_sigmoid", dict(bias=lambda t: t.double())),
    ("route_sigmoid", dict(bias=lambda t: t[:2])),
    ("moe_experts", dict(experts=lambda t: t[:2])), ("moe_experts", dict(rw=lambda t: t[:, :1])), ("moe_experts", dict(x=lambda t: t[:2])),
    ("merged_mlp", dict(x=lambda t: t[:, :8])), ("merged_mlp", dict(up=lambda t: t[:1])),
    ("merged_mlp", dict(down=lambda t: t.transpose(1, 2))), ("merged_mlp", dict(gate=lambda t: t[:, :4])),
    ("combine", dict(cum_ep=lambda t: t[:-1])), ("combine", dict(residual=lambda t: t[:, :8])),
    ("combine", dict(residual=lambda t: t.float())), ("combine", dict(rw=lambda t: t[0]))])
def test_operands_that_a_kernel_would_misread_are_refused(name, changes):
    """Before anything is launched, whatever the device."""
    call, _ = _calls()[name]
    t = _tensors()
    t.update({k: f(t[k]) for k, f in changes.items()})
    with pytest.raises((_n.NativeLibraryError, TypeError), match="expected|must"):
        call(t)


@pytest.mark.parametrize("G,I,H", [(32, 2048, 7168), (32, 256, 1024), (1, 8, 8)])
def test_window_activations_sized_by_a_bound_are_limited(G, I, H):
    """64 MB while nothing is kept for a backward; with one, also a 32nd of the layer's expert weights."""
    f, row = _n.host().sized_by_bound, 2 * (3 * I + H)
    free, kept = (64 << 20) // row, min(64 << 20, 6 * G * I * H // 32) // row
    assert f(free, G, I, H, False) and not f(free + 1, G, I, H, False)
    assert f(kept, G, I, H, True) and not f(kept + 1, G, I, H, True)


class _Hiding(torch.nn.Sequential):
    def named_modules(self, memo=None, prefix="", remove_duplicate=True):
        yield prefix, self
        yield prefix + ".0", self[0]


def _models():
    lin = lambda: torch.nn.Linear(3, 2)
    shared = lin()
    plain = torch.nn.Sequential(lin(), torch.nn.ModuleDict({"a": shared, "b": torch.nn.Sequential(shared, lin())}))
    on_class = _Hiding(lin(), lin())
    inside = torch.nn.Sequential(lin(), _Hiding(lin(), lin()))
    on_itself = torch.nn.Sequential(lin(), lin())
    on_itself.parameters = lambda: iter([on_itself[0].weight])
    stranger = type("Model", (), {"parameters": lambda self: iter(list(plain.parameters())[:3])})()
    return dict(plain=plain, on_class=on_class, inside=inside, on_itself=on_itself, stranger=stranger)


@pytest.mark.parametrize("which", sorted(_models()))
def test_foreign_gradients_are_those_of_the_models_own_traversal(which):
    model = _models()[which]
    params = list(model.parameters())

    def fill(module):                                # (also what an override hides)
        for p in module._parameters.values():
            p.grad = torch.ones_like(p)
        for m in module._modules.values():
            fill(m)
    if isinstance(model, torch.nn.Module):
        fill(model)
    for p in params:
        p.grad = torch.ones_like(p)
    params[0].grad = None
    owned = {id(params[-1])}
    want = [p.grad for p in params if id(p) not in owned and p.grad is not None]
    got = _n.host().foreign_grads(model, owned)
    assert [id(g) for g in got] == [id(g) for g in want]


class _Mlp(torch.nn.Module):
    def __init__(self, make):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = make(), make(), make()


class _Property(torch.nn.Linear):
    @property
    def weight(self):
        return self._parameters["weight"] * 2


class _OwnAccess(torch.nn.Linear):
    def __getattr__(self, name):
        return torch.ones(1) if name == "weight" and "made" in self.__dict__ else super().__getattr__(name)


def _own_access():
    lin = _OwnAccess(3, 2)
    lin.made = True
    return lin


def _shadowed():
    lin = torch.nn.Linear(3, 2)
    lin.__dict__["weight"] = torch.zeros(2, 3)
    return lin


@pytest.mark.parametrize("make", [lambda: torch.nn.Linear(3, 2), _own_access, _shadowed,
                                  lambda: torch.nn.utils.parametrize.register_parametrization(torch.nn.Linear(3, 2), "weight",
                                                                                              torch.nn.Identity())],
                         ids=["plain", "own_access", "on_the_object", "parametrized"])
def test_expert_weights_are_what_attribute_access_gives(make):
    experts = torch.nn.ModuleList([_Mlp(make), _Mlp(lambda: torch.nn.Linear(3, 2)), _Mlp(make)])
    got = _n.host().expert_parameters(experts)
    want = [getattr(e, n).weight for e in experts for n in ("gate_proj", "up_proj", "down_proj")]
    assert len(got) == 9 and all(torch.equal(a, b) for a, b in zip(got, want))
    missing = torch.nn.ModuleList([_Mlp(torch.nn.Identity)])
    with pytest.raises(AttributeError, match="weight"):
        _n.host().expert_parameters(missing)


def test_expert_weights_through_a_property():
    def make():
        lin = _Property.__new__(_Property)
        torch.nn.Module.__init__(lin)
        lin._parameters["weight"] = torch.nn.Parameter(torch.randn(2, 3))
        return lin
    experts = torch.nn.ModuleList([_Mlp(make)])
    got = _n.host().expert_parameters(experts)
    for a, name in zip(got, ("gate_proj", "up_proj", "down_proj")):
        assert torch.equal(a, getattr(experts[0], name)._parameters["weight"] * 2)


def test_row_count_is_waited_for_first_only_where_the_shared_expert_rides():
    """Fewer 128x128 tiles than three quarters of the CUs, the routed experts' extents, dense matrices."""
    f, I, H = _n.host().waits_ahead_of_shared, 1000, 3000

    def shared(i, h):
        return [torch.empty(*s, dtype=torch.bfloat16) for s in ((i, h), (i, h), (h, i))]

    assert f(1000, 32, I, H, 1000, shared(I, H))
    assert f(1000, 32, I, H, 1000, [w.unsqueeze(0) for w in shared(I, H)])
    assert not f(1000, 32, I, H, 1000, shared(2 * I, H))                 # two shared experts as one
    gate, up, down = shared(I, H)
    assert not f(1000, 32, I, H, 1000, [gate, torch.empty(H, I, dtype=torch.bfloat16).t(), down])
    tiles_per_block = (I + 63) // 64
    line = -(-192 // tiles_per_block) * 128                              # 256 CUs
    assert f(1000, 32, I, H, line - 128, shared(I, H)) and not f(1000, 32, I, H, line, shared(I, H))
