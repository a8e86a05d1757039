"""The blocks' autograd nodes (csrc/host/torch_host.cpp) against the contract of a torch.autograd.Function:
in-place changes, saved-tensor hooks, hooks on parameters, repeated backward, threads and streams."""
import collections
import concurrent.futures
import sys
import threading
import time

import pytest
import torch
import torch.nn.utils.parametrize
import torch.utils.checkpoint

pytestmark = pytest.mark.gpu


def _olmoe(merged=True, fp32_logits=True, dtype=torch.bfloat16, H=256, I=256, N=8, K=2):
    from optimus.mapper import ParallelDpPpEpTpMapper
    from optimus.models.common.moe import FastOlmoeParallelSparseMoeBlock
    from optimus.models.olmoe.configuration_olmoe import OlmoeParallelConfig
    cfg = OlmoeParallelConfig(hidden_size=H, intermediate_size=I, num_experts=N, num_experts_per_tok=K, norm_topk_prob=True,
                              use_fast_moe=True, use_merged_mlp_in_fast_moe=merged)
    cfg.router_logits_fp32 = fp32_logits
    return FastOlmoeParallelSparseMoeBlock(cfg, ParallelDpPpEpTpMapper()), dtype


def _dsv3():
    from optimus.mapper import ParallelDpPpEpTpMapper
    from optimus.models.deepseek_v3.configuration_deepseek_v3 import DeepseekV3ParallelConfig
    from optimus.models.deepseek_v3.modeling_deepseek_v3 import DeepseekV3ParallelMoE
    cfg = DeepseekV3ParallelConfig(hidden_size=256, moe_intermediate_size=128, n_routed_experts=16,
                                   num_experts_per_tok=4, n_group=4, topk_group=2, expert_parallelism=2)
    return DeepseekV3ParallelMoE(cfg, ParallelDpPpEpTpMapper(expert_parallelism=2, rank=1)), torch.bfloat16


BLOCKS = {"merged": _olmoe, "per_expert": lambda: _olmoe(merged=False), "model_dtype_logits": lambda: _olmoe(fp32_logits=False),
          "float32": lambda: _olmoe(dtype=torch.float32), "dsv3": _dsv3}


def _block(which, cuda, seed=3):
    torch.manual_seed(seed)
    blk, dtype = BLOCKS[which]()
    for p in blk.parameters():
        torch.nn.init.normal_(p, std=0.05)
    return blk.to(cuda).to(dtype)


def _data(blk, cuda, tokens=192, seed=11):
    g = torch.Generator().manual_seed(seed)
    p = next(blk.parameters())
    return [torch.randn(2, tokens, 256, generator=g).to(p.dtype).to(cuda) for _ in range(2)]


def _out(blk, x):
    out = blk(x)
    return out[0] if isinstance(out, tuple) else out


def _flat_buffers(blk, cuda):
    from optimus.optimizers import MixedPrecisionAdamW
    opt = MixedPrecisionAdamW(blk.parameters(), blk, lr=1e-3, dtype=next(blk.parameters()).dtype, device=cuda)
    opt.zero_grad()
    return opt


# ---- in-place changes of the hidden states -----------------------------------------------------------
@pytest.mark.parametrize("which", sorted(BLOCKS))
@pytest.mark.parametrize("frozen", ["nothing", "gate"])
def test_hidden_states_changed_before_backward_are_refused(cuda, which, frozen):
    """The router hands the hidden states through to the experts; what the experts saved still shares the version
    counter of the caller's tensor.  Nothing may have been added to a live gradient buffer when that is noticed."""
    blk = _block(which, cuda)
    if frozen == "gate":
        blk.gate.requires_grad_(False)
    opt = _flat_buffers(blk, cuda)
    x, d = _data(blk, cuda)
    out = _out(blk, x)
    x.add_(1)
    with pytest.raises(RuntimeError, match="modified (by an )?inplace"):
        out.backward(d)
    assert float(opt.flat_grad.float().abs().max()) == 0.0


def test_router_pass_through_is_a_view_that_cannot_be_changed_in_place(cuda):
    from optimus import _native as _n
    x = torch.randn(64, 512, device=cuda).bfloat16().requires_grad_(True)
    w = torch.randn(8, 512, device=cuda).bfloat16().requires_grad_(True)
    outs = [_n.host().gate_logits(x, w)[1], _n.host().route_softmax(x, w, 2, True, torch.bfloat16, True, False)[3],
            _n.host().route_sigmoid(x, w, torch.zeros(8, device=cuda), 1, 1, 2, True, 1.0)[2]]
    for passed in outs:
        assert passed.data_ptr() == x.data_ptr() and passed._version == x._version
        with pytest.raises(RuntimeError, match="is a view and is being modified inplace"):
            passed.add_(1)


# ---- weights that are not plain parameters ------------------------------------------------------------
class _Doubled(torch.nn.Module):
    def forward(self, w):
        return w * 2


@pytest.mark.parametrize("how", ["parametrized", "plain_tensor"])
def test_merged_weight_that_is_no_parameter(cuda, how):
    """w * 2 in the place of every merged expert weight: the block of doubled weights, gradients reaching w."""
    names = ("gate_proj_merged_weight", "up_proj_merged_weight", "down_proj_merged_weight")
    blk, plain = _block("merged", cuda), _block("merged", cuda)
    with torch.no_grad():
        for n in names:
            getattr(plain.experts, n).mul_(2)
    leaves = []
    for n in names:
        w = getattr(blk.experts, n)
        if how == "parametrized":
            torch.nn.utils.parametrize.register_parametrization(blk.experts, n, _Doubled())
            leaves.append(blk.experts.parametrizations[n].original)
        else:
            delattr(blk.experts, n)
            setattr(blk.experts, n, w * 2)
            leaves.append(w)
    x, d = _data(blk, cuda)
    a, b = _out(blk, x), _out(plain, x)
    assert torch.equal(a, b)
    a.backward(d)
    b.backward(d)
    for n, w in zip(names, leaves):
        assert torch.equal(w.grad, getattr(plain.experts, n).grad * 2), n


# ---- saved tensors ------------------------------------------------------------------------------------
def _grads_of(blk, x):
    return [x.grad] + [p.grad for p in blk.parameters()]


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_backward_computes_with_what_saved_tensor_hooks_unpack(cuda, which):
    """Everything saved is packed to the host; x, every weight and the routing change before the backward, which
    must give the gradients of the values at the time of the forward."""
    ref, blk = _block(which, cuda), _block(which, cuda)
    x, d = _data(blk, cuda)
    xr, xb = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    _out(ref, xr).backward(d)
    packed = []

    def pack(t):
        packed.append(t.data_ptr())
        return t.detach().to("cpu", copy=True)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(cuda)):
        out = _out(blk, xb)
    weights = [p for n, p in blk.named_parameters()]
    assert {w.data_ptr() for w in weights if w.dim() == 3} <= set(packed)
    with torch.no_grad():
        for w in weights + [xb]:
            w.mul_(-3)
    out.backward(d)
    for a, b in zip(_grads_of(blk, xb), _grads_of(ref, xr)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("which,name", [("merged", "experts.up_proj_merged_weight"), ("per_expert", "experts.5.down_proj.weight"),
                                        ("dsv3", "experts.7.gate_proj.weight"), ("dsv3", "shared_experts.up_proj.weight"),
                                        ("float32", "experts.down_proj_merged_weight")])
def test_weight_changed_before_backward_is_refused(cuda, which, name):
    blk = _block(which, cuda)
    x, d = _data(blk, cuda)
    out = _out(blk, x)
    with torch.no_grad():
        dict(blk.named_parameters())[name].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(d)


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_second_backward_is_refused_or_repeats(cuda, which):
    blk = _block(which, cuda)
    opt = _flat_buffers(blk, cuda)
    x, d = _data(blk, cuda)
    out = _out(blk, x)
    out.backward(d, retain_graph=True)
    once = opt.flat_grad.clone()
    opt.zero_grad()
    out.backward(d)
    assert torch.equal(opt.flat_grad, once) and float(once.float().abs().max()) > 0
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(d)
    assert torch.equal(opt.flat_grad, once)


@pytest.mark.parametrize("which", ["merged", "model_dtype_logits", "float32", "dsv3"])
def test_gate_weight_of_any_strides(cuda, which):
    blk, ref = _block(which, cuda), _block(which, cuda)
    gate = blk.gate
    gate.weight = torch.nn.Parameter(gate.weight.detach().t().contiguous().t())
    assert not gate.weight.is_contiguous()
    x, d = _data(blk, cuda)
    a, b = _out(blk, x), _out(ref, x)
    assert torch.equal(a, b)
    a.backward(d)
    b.backward(d)
    assert torch.equal(gate.weight.grad, ref.gate.weight.grad)


# ---- hooks on parameters ------------------------------------------------------------------------------
@pytest.mark.parametrize("which,name", [("merged", "experts.gate_proj_merged_weight"), ("per_expert", "experts.3.up_proj.weight"),
                                        ("dsv3", "shared_experts.down_proj.weight")])
@pytest.mark.parametrize("kind", ["tensor", "post_accumulate"])
def test_parameter_hooks_see_the_gradient_while_they_are_registered(cuda, which, name, kind):
    """A live hook gets the gradient of this pass; once it is removed the GEMMs add into the buffer in place again,
    as they do for a parameter whose hook dictionary a deepcopy left empty."""
    from optimus import _native as _n
    blk = _block(which, cuda)
    opt = _flat_buffers(blk, cuda)
    p = dict(blk.named_parameters())[name]
    x, d = _data(blk, cuda)
    _out(blk, x).backward(d)
    want = p.grad.clone()
    seen = []
    if kind == "tensor":
        handle = p.register_hook(lambda g: seen.append(g.clone()))
    else:
        handle = p.register_post_accumulate_grad_hook(lambda q: seen.append(q.grad.clone()))
    opt.zero_grad()
    assert _n.host().live_grad(p) is None
    _out(blk, x).backward(d)
    assert len(seen) == 1 and torch.equal(seen[0], want) and torch.equal(p.grad, want)
    handle.remove()
    copied = torch.nn.Parameter(p.detach().clone())
    copied._backward_hooks = collections.OrderedDict()
    copied.grad = torch.zeros(2 * p.numel(), device=cuda, dtype=p.dtype)[:p.numel()].view_as(p)
    for q in (p, copied):
        assert _n.host().live_grad(q).data_ptr() == q.grad.data_ptr()
    _n.launch_log = []
    try:
        opt.zero_grad()
        _out(blk, x).backward(d)
    finally:
        names, _n.launch_log = [e[0] for e in _n.launch_log], None
    assert sum("wgrad" in n and n.startswith("om_grouped") and not n.endswith("accumulate") for n in names) == 0
    assert len(seen) == 1 and torch.equal(p.grad, want)


# ---- Python code called from the host module ----------------------------------------------------------
@pytest.mark.parametrize("which", ["merged", "float32", "dsv3"])
@pytest.mark.parametrize("where", ["start", "stop"])
@pytest.mark.parametrize("direction", ["forward", "backward"])
def test_an_exception_of_the_profiler_reaches_the_caller(cuda, which, where, direction):
    import optimus.globals
    from optimus.profilers import PclProfiler

    class Failing(PclProfiler):
        armed = False

        def start(self, name, key=""):
            if self.armed and where == "start":
                raise LookupError("profiler start")
            super().start(name, key)

        def stop(self, name):
            super().stop(name)
            if self.armed and where == "stop":
                raise LookupError("profiler stop")

    blk = _block(which, cuda)
    x, d = _data(blk, cuda)
    want = _out(blk, x)
    prof = Failing()
    optimus.globals.profiler = prof
    try:
        _out(blk, x).backward(d)                 # (registers the timers: an unknown one would fail in its turn)
        prof.armed = direction == "forward"
        if direction == "forward":
            with pytest.raises(LookupError, match="profiler " + where):
                _out(blk, x)
        else:
            out = _out(blk, x)
            prof.armed = True
            with pytest.raises(LookupError, match="profiler " + where):
                out.backward(d)
    finally:
        optimus.globals.profiler = None
    assert torch.equal(_out(blk, x), want)       # and the module goes on


def test_an_exception_of_the_launch_log_reaches_the_caller(cuda, monkeypatch):
    from optimus import _native as _n
    blk = _block("merged", cuda)
    x, d = _data(blk, cuda)
    out = _out(blk, x)

    def fail(*a):
        raise LookupError("log")
    for name in ("timed_begin", "timed_end"):
        with monkeypatch.context() as m:
            m.setattr(_n, name, fail)
            m.setattr(_n, "launch_log", [])
            with pytest.raises(LookupError):
                _out(blk, x)
            with pytest.raises(LookupError):
                out.backward(d, retain_graph=True)
    out.backward(d)


# ---- threads and streams ------------------------------------------------------------------------------
def test_forward_calls_let_other_python_threads_run(cuda):
    """With the interpreter's own switching out of the way, another thread only runs where a call lets the GIL go."""
    from optimus import _native as _n
    experts = torch.zeros(512, 8, dtype=torch.int64, device=cuda)
    call = _n.host().build_token_permutation
    call(experts, 0, 8)
    ticks, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            time.sleep(0)                        # (lets the GIL go and asks for it again)
            ticks[0] += 1
    t = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000)
    try:
        t.start()
        time.sleep(0.01)
        before, kept = ticks[0], []              # (kept: freeing a tensor would let the GIL go too)
        while ticks[0] == before and len(kept) < 2000:
            kept.append(call(experts, 0, 8))
        assert ticks[0] > before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        t.join()


@pytest.mark.parametrize("which", ["merged", "per_expert", "dsv3", "float32"])
def test_threads_with_streams_of_their_own(cuda, which):
    """Four threads, each a block, a stream and inputs of its own: the gradients of a single thread."""
    def work(seed, stream):
        with torch.cuda.stream(stream):
            blk = _block_cache[seed]
            res = []
            for i in range(6):
                x, d = _block_data[seed]
                xi = x.clone().requires_grad_(True)
                for p in blk.parameters():
                    p.grad = None
                out = _out(blk, xi)
                out.backward(d)
                res = [out.detach()] + _grads_of(blk, xi)
            stream.synchronize()
            return res
    seeds = range(4)
    _block_cache = {s: _block(which, cuda, seed=s) for s in seeds}
    _block_data = {s: _data(_block_cache[s], cuda, seed=s) for s in seeds}
    torch.cuda.synchronize()
    want = [work(s, torch.cuda.current_stream()) for s in seeds]
    streams = [torch.cuda.Stream() for _ in seeds]
    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        got = list(pool.map(work, seeds, streams))
    for a, b in zip(got, want):
        for u, v in zip(a, b):
            assert torch.equal(u, v)


@pytest.mark.parametrize("which", ["merged", "dsv3"])
def test_two_threads_run_backward_through_one_graph(cuda, which):
    """Eight passes from four threads through one retained graph, then a pass that releases it beside another: the
    gradients of one pass each, and in the end the refusal of a second backward, nothing else."""
    blk = _block(which, cuda)
    x, d = _data(blk, cuda)
    x.requires_grad_(True)
    inputs = [x] + list(blk.parameters())
    out = _out(blk, x)
    want = torch.autograd.grad(out, inputs, d, retain_graph=True)
    grad = lambda retain: torch.autograd.grad(out, inputs, d, retain_graph=retain)
    torch.cuda.synchronize()
    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        for got in pool.map(grad, [True] * 8):
            for u, v in zip(got, want):
                assert torch.equal(u, v)
        ends = [pool.submit(grad, False) for _ in range(4)]
    done = 0
    for e in ends:
        err = e.exception()
        assert err is None or "second time" in str(err), err
        done += err is None
    assert done >= 1


# ---- the public autograd functions beside the nodes ---------------------------------------------------
def _grad_results(outs, inputs, seed=5):
    g = torch.Generator().manual_seed(seed)
    outs = [o for o in outs if o.requires_grad]
    ds = [torch.randn(o.shape, generator=g).to(o.dtype).to(o.device) for o in outs]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, inputs, ds))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_router_functions_equal_the_nodes(cuda, dtype):
    from optimus import _native as _n
    from optimus.models.common import moe
    g = torch.Generator().manual_seed(0)
    x = torch.randn(300, 512, generator=g).to(dtype).to(cuda).requires_grad_(True)
    w = (torch.randn(8, 512, generator=g) * 0.05).to(dtype).to(cuda).requires_grad_(True)
    pairs = [(lambda: moe.GateLogitsFunction.apply(x, w), lambda: _n.host().gate_logits(x, w))]
    if dtype == torch.float32:
        pairs.append((lambda: [moe.GateLogitsF32Function.apply(x, w)], lambda: [_n.host().gate_logits(x, w)[0]]))
    pairs.append((lambda: moe.GateSoftmaxTopkFunction.apply(x, w, 2, True, dtype),
                  lambda: _n.host().route_softmax(x, w, 2, True, dtype, True, False)))
    for ours, node in pairs:
        for a, b in zip(_grad_results(ours(), [x, w]), _grad_results(node(), [x, w])):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("live", [False, True])
def test_expert_functions_equal_the_nodes(cuda, dtype, live):
    """Merged and per-expert weights, gathered and not, fresh gradients and live ones."""
    from optimus import _native as _n
    from optimus.models.common import moe
    T, K, G, H, I = 100, 2, 4, 64, 72
    g = torch.Generator().manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda)
    experts = torch.randint(0, G, (T, 1), generator=g) + torch.arange(K)
    cum, cum_ep, rows, out_rows, sel = moe.build_token_permutation((experts % G).to(cuda), 0, G)
    x = rnd(T, H).to(dtype).requires_grad_(True)
    rw = rnd(T, K).abs().to(dtype).requires_grad_(True)
    res = rnd(T, H).to(dtype).requires_grad_(True)
    merged = [(rnd(G, o, i) * 0.1).to(dtype).requires_grad_(True) for o, i in ((I, H), (I, H), (H, I))]
    bank = [m.detach().clone() for m in merged]
    each = [bank[j][n].detach().requires_grad_(True) for n in range(G) for j in range(3)]
    shared = [(rnd(o, i) * 0.1).to(dtype).requires_grad_(True) for o, i in ((I, H), (I, H), (H, I))]
    one = moe.single_segment_counts(T, cuda)
    host = _n.host()
    gathered = (rows, cum_ep, out_rows)
    cases = {   # (function, node, activations, weights)
        "merged": (lambda v: moe.MergedMLPFunction.apply(v, *merged, cum), lambda v: host.merged_mlp(v, cum, True, merged, None, None, None), merged),
        "per_expert": (lambda v: moe.GroupMLPFunction.apply(v, cum, False, *each), lambda v: host.merged_mlp(v, cum, False, each, None, None, None), each),
        "single": (lambda v: moe.MergedMLPFunction.apply(v, *shared, moe.single_segment_counts(v.shape[0], cuda)),
                   lambda v: host.merged_mlp(v, moe.single_segment_counts(v.shape[0], cuda), True, shared, None, None, None), shared),
        "gathered": (lambda v: moe.GatheredMergedMLPFunction.apply(x, *gathered, *merged, cum), lambda v: host.merged_mlp(x, cum, True, merged, *gathered), merged),
        "gathered_per_expert": (lambda v: moe.GatheredGroupMLPFunction.apply(x, *gathered, cum, *each),
                                lambda v: host.merged_mlp(x, cum, False, each, *gathered), each)}
    xg = x.detach()[rows.long()].requires_grad_(True)
    y = rnd(T * K, H).to(dtype).requires_grad_(True)
    combine = {"combine": (moe.GroupGemmOutputReductionFunction, None, [y, rw]),
               "combine_residual": (moe.GroupGemmOutputReductionResidualFunction, res, [y, rw, res])}

    def results(out, acts, weights):
        if not live:
            return _grad_results([out], acts + list(weights))
        for w in weights:                        # (several weights in one buffer: per-expert sinks need a constant pitch)
            w.grad = None
        if len(weights) == 3 * G:
            for j in range(3):
                buf = torch.ones(2, G, *weights[j].shape, device=cuda, dtype=dtype)[0]
                for n in range(G):
                    weights[3 * n + j].grad = buf[n]
        else:
            for w in weights:
                w.grad = torch.ones(2, *w.shape, device=cuda, dtype=dtype)[0]
        kept = [w.grad for w in weights]
        for a in acts:
            a.grad = None
        out.backward(torch.ones_like(out) * 0.5)
        assert all(w.grad is k for w, k in zip(weights, kept))
        return [out.detach()] + [a.grad for a in acts] + [w.grad.clone() for w in weights]

    for name, (ours, node, weights) in cases.items():
        act = x if name.startswith("gathered") else xg
        for a, b in zip(results(ours(act), [act], weights), results(node(act), [act], weights)):
            assert torch.equal(a, b), name
    for name, (cls, residual, ins) in combine.items():
        extra = () if residual is None else (residual,)
        for a, b in zip(_grad_results([cls.apply(y, rw, cum_ep, sel, rows, out_rows, *extra)], ins),
                        _grad_results([host.combine(y, rw, cum_ep, sel, rows, out_rows, residual)], ins)):
            assert torch.equal(a, b), name
    if dtype == torch.float32:
        return
    routed = {
        "routed": (lambda: moe.RoutedMLPFunction.apply(x, rw, rows, cum_ep, out_rows, sel, cum, res, True, *merged),
                   lambda: host.moe_experts(x, rw, (experts % G).to(cuda), 0, G, G, False, res, True, merged, False, None),
                   [x, rw, res], merged),
        "routed_per_expert": (lambda: moe.RoutedMLPFunction.apply(x, rw, rows, cum_ep, out_rows, sel, cum, None, False, *each),
                              lambda: host.moe_experts(x, rw, (experts % G).to(cuda), 0, G, G, False, None, False, each, False, None),
                              [x, rw], each)}
    for name, (ours, node, acts, weights) in routed.items():
        for a, b in zip(results(ours(), acts, weights), results(node(), acts, weights)):
            assert torch.equal(a, b), name
    for w in each + shared:
        w.grad = None
    both = lambda f: _grad_results([f], [x, rw] + each + shared)
    for a, b in zip(both(moe.RoutedAndSharedMLPFunction.apply(x, rw, rows, cum_ep, out_rows, sel, cum, False, *each, *shared)),
                    both(host.moe_experts(x, rw, (experts % G).to(cuda), 0, G, G, False, None, False, each + shared, True, one))):
        assert torch.equal(a, b)


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_forward_mode_through_a_block_is_refused(cuda, which):
    blk = _block(which, cuda)
    x, d = _data(blk, cuda)
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
        _out(blk, torch.autograd.forward_ad.make_dual(x, d))


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_only_a_pass_that_accumulates_adds_into_live_gradients(cuda, which):
    """torch.autograd.grad returns gradients and leaves .grad alone; backward(inputs=...) adds only where it is told."""
    blk = _block(which, cuda)
    opt = _flat_buffers(blk, cuda)
    x, d = _data(blk, cuda)
    x.requires_grad_(True)
    params = list(blk.parameters())
    out = _out(blk, x)
    out.backward(d, retain_graph=True)
    want = [p.grad.clone() for p in params]
    dx = x.grad.clone()
    opt.zero_grad()
    got = torch.autograd.grad(out, [x] + params, d, retain_graph=True)
    only_x = torch.autograd.grad(out, x, d, retain_graph=True)[0]
    assert float(opt.flat_grad.float().abs().max()) == 0.0
    for a, b in zip(got, [dx] + want):
        assert torch.equal(a, b)
    assert torch.equal(only_x, dx)
    out.backward(d, inputs=[params[1]])
    for i, p in enumerate(params):
        assert torch.equal(p.grad, want[i] if i == 1 else torch.zeros_like(p))


def test_a_training_step_keeps_no_activations_of_other_ranks_pairs(cuda):
    """An expert window of 8 of 16 experts: what a forward pass keeps for backward is sized by the rows routed here
    (the bound would be over twice that), a forward without gradients may use the bound."""
    blk = _block("dsv3", cuda)
    x, _ = _data(blk, cuda, tokens=1024)
    with torch.no_grad():
        experts, _w = blk.gate(x)
    here = int((experts >= 8).sum())
    T, H, I = 2048, 256, 128
    x.requires_grad_(True)
    _out(blk, x)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = _out(blk, x)
    kept = torch.cuda.memory_allocated() - before
    # g, u, h of the routed and the shared expert, the output, routing and index arrays (T rows of 16 + 6 * 4 words)
    assert kept <= 1.1 * (2 * 3 * I * (here + T) + 2 * T * H + 4 * T * 64) < 2 * 3 * I * (4 * T + T)
    del out


# ---- activation checkpointing around a block ----------------------------------------------------------
@pytest.mark.parametrize("which", sorted(BLOCKS))
@pytest.mark.parametrize("reentrant", [False, True])
def test_checkpointed_region_around_a_block(cuda, which, reentrant):
    """torch's layers before the block in one checkpointed region: the recomputation starts when the block's node
    unpacks what it saved, and has to record those layers too."""
    blk = _block(which, cuda)
    dtype = next(blk.parameters()).dtype
    torch.manual_seed(1)
    before = torch.nn.Sequential(torch.nn.Linear(256, 256, bias=False), torch.nn.GELU(), torch.nn.LayerNorm(256)).to(cuda).to(dtype)
    x, d = _data(blk, cuda)
    region = lambda v: _out(blk, before(v))
    params = list(before.parameters()) + list(blk.parameters())

    def grads(f):
        v = x.clone().requires_grad_(True)
        for p in params:
            p.grad = None
        out = f(v)
        out.backward(d)
        return [out.detach(), v.grad] + [p.grad for p in params]
    want = grads(region)
    got = grads(lambda v: torch.utils.checkpoint.checkpoint(region, v, use_reentrant=reentrant))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_callers_stream_waits_for_gradients_added_in_place(cuda, which):
    """Forward on a side stream that is busy, backward called from the current one, no gradient but the in-place ones:
    what the caller's stream reads next is the finished sum."""
    blk = _block(which, cuda)
    blk.gate.requires_grad_(False)
    opt = _flat_buffers(blk, cuda)
    x, d = _data(blk, cuda)
    other = _out(blk, x)                             # (keeps the parameters' accumulation nodes on this stream)
    _out(blk, x).backward(d)
    want = opt.flat_grad.clone()
    opt.zero_grad()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = _out(blk, x)
        torch.cuda._sleep(100_000_000)               # (some 50 ms)
    out.backward(d)
    got = opt.flat_grad.clone()
    torch.cuda.synchronize()
    assert torch.equal(got, want) and float(want.float().abs().max()) > 0
    del other
