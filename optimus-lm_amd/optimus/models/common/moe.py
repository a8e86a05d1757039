"""optimus.models.common.moe — the fast MoE block, same interface as the reference
(optimus/models/common/moe.py:43-632), computed by the HIP kernels of liboptimus_mi355x.so.

Pipeline of FastOlmoeParallelSparseMoeBlock.forward (reference moe.py:454-621):
  router (softmax -> top-K -> optional renorm)     one wavefront per token          [route.hip]
  K1+K2+K3 index construction                      stable counting sort on device   [sort.hip]
  K4 gather rows into expert order                                                   [rows.hip]
  K5 merged-MLP grouped SwiGLU GEMMs               bf16 MFMA, variable rows/expert  [ggemm.hip]
  K6 weighted combine back to token order                                            [rows.hip]
and the mirrored backward.  There is one code path: the reference's `use_triton_path_*` and
`use_ref_path_*` switches are accepted where its signatures have them and ignored.
"""
import functools
import warnings

import torch
import torch.nn as nn
from torch.utils.checkpoint import checkpoint as torch_activation_checkpoint

import pcl_xpu_customops
from optimus import _native as _n
from optimus.profilers import record_pcl_function


# Two of the blocks' fusions only take some operands (see gate_kernel_fits, routed_mlp_kernel_fits);
# for the others the same block runs its unfused sequence of kernels from this library, whose bf16
# roundings fall in other places.  That switch is announced once per reason (a UserWarning), or
# refused when strict_fused_paths is set.
strict_fused_paths = False
_announced_switches = set()


def note_unfused_path(what, why, instead="running the unfused sequence of kernels (same mathematics, bf16 "
                                            "roundings in other places)"):
    """Called where a block leaves a fused kernel path for the unfused sequence."""
    if (what, why) in _announced_switches and not strict_fused_paths:
        return
    message = f"{what}: {why}; {instead}"
    if strict_fused_paths:
        raise _n.NativeLibraryError(message + " [strict_fused_paths is set]")
    _announced_switches.add((what, why))
    warnings.warn(message, stacklevel=3)


def get_tensor_list(tensor, cum_token_counts):
    """Per-expert row slices (reference moe.py:28-35); host-side helper, needs CPU-readable counts."""
    N = len(cum_token_counts) - 1
    return [tensor[cum_token_counts[n]:cum_token_counts[n + 1]] for n in range(N)]


def _device_counts(cum_token_counts, device):
    """The reference hands MergedMLP a CPU int32 tensor (moe.py:494); the kernels read the counts
    from device memory, so accept either and never read them back."""
    if cum_token_counts.device != device:
        cum_token_counts = cum_token_counts.to(device, non_blocking=True)
    if cum_token_counts.dtype != torch.int32:
        cum_token_counts = cum_token_counts.to(torch.int32)
    return cum_token_counts.contiguous()


_single_segment_cache = {}


def single_segment_counts(rows, device):
    """cum_token_counts of one expert that owns all `rows` rows: the device int32 tensor [0, rows],
    built once per (rows, device) so that a dense MLP run through the grouped kernels copies nothing
    from the host per call.  Read-only by contract."""
    key = (int(rows), str(device))
    cum = _single_segment_cache.get(key)
    if cum is None:
        if len(_single_segment_cache) >= 64:
            _single_segment_cache.clear()
        cum = _single_segment_cache[key] = torch.tensor([0, int(rows)], dtype=torch.int32, device=device)
    return cum


def _expert_stride(weight):
    """Elements between consecutive experts of a [G, out, in] weight whose inner two dims are
    dense; 0 for the packed layout."""
    G, o, i = weight.shape
    if weight.stride(2) != 1 or weight.stride(1) != i:
        raise _n.NativeLibraryError("expert weights must be dense [out, in] matrices")
    s = weight.stride(0) if G > 1 else o * i
    return 0 if s == o * i else s


def _require_bf16(*tensors):
    for t in tensors:
        if t.dtype != torch.bfloat16:
            raise TypeError(f"the fused expert kernels run in bfloat16 (got {t.dtype}); cast the "
                            "module with .to(torch.bfloat16)")


def _gemm_dtype(*tensors):
    """bfloat16 (the tuned kernels) or float32 (the plain fp32 kernels) for all operands."""
    dt = tensors[0].dtype
    if dt not in (torch.bfloat16, torch.float32) or any(t.dtype != dt for t in tensors):
        raise TypeError("the grouped expert GEMMs take operands that are all bfloat16 or all float32 "
                        f"(got {[str(t.dtype) for t in tensors]})")
    return dt


def _grouped_gemm(kind, a, b, out, cum, rows, G, N, K, w_stride, accumulate=False):
    """om_grouped_gemm_{fwd,dgrad,wgrad}[_f32][_accumulate] by the operands' dtype; `accumulate`
    (wgrad only) adds the product to `out` in place."""
    suffix = "_f32" if _gemm_dtype(a, b, out) == torch.float32 else ""
    name = f"om_grouped_gemm_{kind}{suffix}" + ("_accumulate" if accumulate else "")
    _n.check(getattr(_n.lib(), name)(_n.ptr(a), _n.ptr(b), _n.ptr(out), _n.ptr(cum), rows, G, N, K,
                                     w_stride, _n.stream()), name)


# ----------------------------------------------------------------------------------------------
# Router
# ----------------------------------------------------------------------------------------------
def gate_kernel_unfit_reason(x, weight):
    """None when the fused gate + routing kernel (om_router_gate_softmax_topk) takes these operands,
    else why not.  (om_router_gate_split_softmax_topk takes the others; for small gates, up to 64 experts
    and 65536 weights, that is one launch too, but not this kernel.)"""
    if not (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16):
        return f"operands are not bfloat16 device tensors ({x.dtype}, {weight.dtype})"
    N, H = weight.shape
    if N > 256:
        return f"{N} experts (the kernel takes at most 256)"
    if x.shape[0] == 0:
        return "no tokens"
    need = 512 if N <= 64 else 256 if N <= 128 else 64
    if H % need != 0:
        return f"hidden size {H} is not a multiple of {need} (needed with {N} experts)"
    return None


def gate_kernel_fits(x, weight):
    """Shapes and dtypes the fused gate + routing kernel takes (om_router_gate_softmax_topk)."""
    return gate_kernel_unfit_reason(x, weight) is None


def _require_gate_shape(weight, h_multiple, what):
    N, H = weight.shape
    if N > 256 or H % h_multiple != 0:
        raise _n.NativeLibraryError(
            f"{what}: the gate kernels take at most 256 experts and hidden sizes that are multiples "
            f"of {h_multiple} (got {N} experts, hidden {H}); there is no library fallback")


def _gate_weight_grad(x, weight, dlogits):
    """dweight[n,h] = sum_t dlogits[t,n] x[t,h]: a long contraction with a tiny output, split
    over token ranges on the device (om_router_gate_wgrad) instead of a library GEMM that would
    run on a few CUs."""
    return _n.host().gate_weight_grad(x, weight, dlogits)


def _gate_input_grad(weight, dlogits, other_grad=None):
    """dx = bf16(dlogits) @ weight (om_router_gate_dgrad).  With `other_grad` [T,H] (the gradient
    that reached the same hidden states through the experts) the sum of the two is returned, formed
    inside the kernel with autograd's two roundings, so no separate accumulation pass runs."""
    return _n.host().gate_input_grad(weight, dlogits, other_grad)


def _gate_backward(x, weight, dlogits, needs, other_grad=None):
    """(dx, dweight) of logits = x @ weight.T for a bf16 gate from the fp32 gradient of the logits,
    rounded to bf16 as it is loaded (the precision a bf16 router's backward has anyway), both on
    bf16 MFMA with fp32 accumulation: om_router_gate_dgrad and om_router_gate_wgrad.  `other_grad`
    is added to dx inside the kernel (see _gate_input_grad)."""
    _require_bf16(x, weight)
    return _n.host().gate_backward(x, weight, dlogits, needs[0], needs[1], other_grad)


def fp32_logits_with_passthrough(x, weight):
    """(router logits in float32, x) from 2-D x [T,H] and weight [N,H] (the gate's nn.Linear weight).
    bf16 operands go through the gate kernels (at most 256 experts, H a multiple of 8; anything
    else raises), a float32 module's on the plain float32 gate kernels.  The second result is the input
    itself; a caller that feeds the rest of the layer from it makes that part's input gradient arrive at
    the gate, where the gate's own is added to it."""
    if x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16:
        # (the forward and the two backward kernels take the same shapes, so a shape that passes here
        # passes in backward)
        _require_gate_shape(weight, 8, "gate projection")
        return _n.host().gate_logits(x.contiguous(), weight.contiguous())
    if x.dtype == torch.float32 and weight.dtype == torch.float32:
        return _n.host().gate_logits(x.contiguous(), weight.contiguous())
    raise TypeError(f"router gate: activations and weight must both be bfloat16 or both float32 "
                    f"(got {x.dtype}, {weight.dtype})")


def fp32_logits(x, weight):
    """Router logits in float32 (see fp32_logits_with_passthrough)."""
    return fp32_logits_with_passthrough(x, weight)[0]


def gate_logits(x, gate):
    """router_logits = gate(x) in the module's dtype (reference moe.py:456,
    modeling_olmoe.py:284) for 2-D x.  A bf16 gate runs on the gate kernels: the fp32-accumulated
    logits rounded once to bf16, which is what a bf16 linear layer returns (up to the order of the
    fp32 sum).  A float32 module's gate runs on the plain float32 gate kernels."""
    return gate_logits_with_passthrough(x, gate)[0]


def gate_logits_with_passthrough(x, gate):
    """(gate_logits(x, gate), x), the second being the gate kernels' pass-through of x for a bf16
    gate (see fp32_logits_with_passthrough) and x itself otherwise."""
    if x.dtype == torch.bfloat16 and gate.weight.dtype == torch.bfloat16:
        logits, x = fp32_logits_with_passthrough(x, gate.weight)
        return logits.to(torch.bfloat16), x
    if x.dtype == torch.float32 and gate.weight.dtype == torch.float32 and x.is_cuda and gate.bias is None:
        return fp32_logits_with_passthrough(x, gate.weight)
    return gate(x), x


# The autograd functions below wrap the same kernels, in the same order, as the C++ nodes that the blocks use
# (csrc/host/torch_host.cpp: gate_logits, route_softmax, merged_mlp, moe_experts, combine): for callers that apply
# or extend the reference's functions one by one.
class GateLogitsFunction(torch.autograd.Function):
    """(fp32 logits, x) of the gate projection.  The second output is the input itself; a caller that
    feeds the rest of the layer from it makes that part's input gradient arrive here, where the gate's
    own is added to it inside the input-gradient kernel instead of by a separate accumulation pass."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.save_for_backward(x, weight)
        ctx.set_materialize_grads(False)
        return _n.host().gate_logits(x, weight)

    @staticmethod
    def backward(ctx, dlogits, x_grad):
        if dlogits is None:
            return x_grad, None
        return _n.host().gate_backward(*ctx.saved_tensors, dlogits, *ctx.needs_input_grad, x_grad)


class GateLogitsF32Function(torch.autograd.Function):
    """logits = x @ weight.T for a float32 gate (om_router_gate_logits_f32, with both backward products
    on the float32 gate kernels)."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.save_for_backward(x, weight)
        return _n.host().gate_logits(x, weight)[0]

    @staticmethod
    def backward(ctx, dlogits):
        return _n.host().gate_backward(*ctx.saved_tensors, dlogits, *ctx.needs_input_grad, None)


class GateSoftmaxTopkFunction(torch.autograd.Function):
    """The OLMoE router with the gate projection: fp32 logits, softmax, top-K, optional renormalisation,
    in one launch (om_router_gate_softmax_topk) or, up to 2048 tokens, in two with the same bits
    (om_router_gate_split_softmax_topk).  Returns (routing_weights, selected_experts, router_logits fp32,
    hidden_states); reference moe.py:456 and :467-471.

    The fourth output is the input itself.  A caller that feeds the experts from it (instead of from
    the tensor it passed in) makes the experts' input gradient arrive here, where the gate's own
    input gradient is added to it inside om_router_gate_dgrad: one pass over [T,H] instead of a
    matmul output plus autograd's accumulation kernel."""

    @staticmethod
    def forward(ctx, x, weight, top_k, norm_topk_prob, out_dtype):
        weights, experts, logits, passed = _n.host().route_softmax(x, weight, top_k, bool(norm_topk_prob), out_dtype,
                                                                   True, False)
        ctx.save_for_backward(x, weight, logits, experts)
        ctx.norm_topk_prob = bool(norm_topk_prob)
        ctx.mark_non_differentiable(experts)
        # an output nobody differentiates (the logits without an auxiliary loss) arrives as None in
        # backward instead of a tensor of zeros that would have to be filled and added
        ctx.set_materialize_grads(False)
        return weights, experts, logits, passed

    @staticmethod
    def backward(ctx, weights_grad, _experts_grad, logits_grad, x_grad):
        x, weight, logits, experts = ctx.saved_tensors
        if weights_grad is None and logits_grad is None:
            return x_grad, None, None, None, None
        dlogits = logits_grad
        if weights_grad is not None:
            dlogits = _softmax_topk_backward(logits, experts, weights_grad, ctx.norm_topk_prob)
            if logits_grad is not None:
                dlogits = dlogits + logits_grad
        dx, dw = _n.host().gate_backward(x, weight, dlogits, *ctx.needs_input_grad[:2], x_grad)
        return dx, dw, None, None, None


def _softmax_topk_backward(router_logits, experts, weights_grad, norm_topk_prob):
    """Gradient of the logits of a softmax top-K router."""
    T, N = router_logits.shape
    weights_grad = weights_grad.contiguous()
    dlogits = torch.empty_like(router_logits)
    _n.check(_n.lib().om_route_softmax_topk_bwd(
        _n.ptr(router_logits), _n.dtype_code(router_logits), _n.ptr(experts), _n.ptr(weights_grad),
        _n.dtype_code(weights_grad), T, N, experts.shape[1], int(norm_topk_prob), _n.ptr(dlogits),
        _n.stream()), "om_route_softmax_topk_bwd")
    return dlogits


class SoftmaxTopkRouterFunction(torch.autograd.Function):
    """routing_weights, selected_experts = topk(softmax_fp32(logits), K) [/ sum] -> out dtype.

    Reference moe.py:467-471.  Selection order is (probability desc, expert index asc)."""

    @staticmethod
    def forward(ctx, router_logits, top_k, norm_topk_prob, out_dtype):
        _n.require_cuda_contiguous(router_logits)
        T, N = router_logits.shape
        weights = torch.empty((T, top_k), dtype=out_dtype, device=router_logits.device)
        experts = torch.empty((T, top_k), dtype=torch.int64, device=router_logits.device)
        _n.check(_n.lib().om_route_softmax_topk(
            _n.ptr(router_logits), _n.dtype_code(router_logits), T, N, top_k, int(bool(norm_topk_prob)),
            _n.ptr(weights), _n.dtype_code(weights), _n.ptr(experts), _n.stream()),
            "om_route_softmax_topk")
        ctx.save_for_backward(router_logits, experts)
        ctx.norm_topk_prob = bool(norm_topk_prob)
        ctx.mark_non_differentiable(experts)
        return weights, experts

    @staticmethod
    def backward(ctx, weights_grad, _experts_grad):
        dlogits = _softmax_topk_backward(*ctx.saved_tensors, weights_grad, ctx.norm_topk_prob)
        return dlogits, None, None, None


# ----------------------------------------------------------------------------------------------
# Index construction (K1 + K2 + K3)
# ----------------------------------------------------------------------------------------------
def build_token_permutation(selected_experts, expert_start_idx, expert_end_idx):
    """Stable counting sort of the (token, k) pairs routed to [expert_start_idx, expert_end_idx).

    Returns device int32 tensors (cum_token_counts [NR+1], cum_expert_counts_ep [T+1],
    input_indices, output_indices, selected_experts_indices) — the last three sized T*K; only
    the first cum_token_counts[-1] entries are meaningful.  Same values as the reference's
    K1 -> cumsum -> K3 sequence (moe.py:499-554).  Nothing is copied to the host."""
    return _n.host().build_token_permutation(selected_experts, int(expert_start_idx), int(expert_end_idx))


# ----------------------------------------------------------------------------------------------
# Weight gradients accumulated in place
# ----------------------------------------------------------------------------------------------
# The reference trains with every p.grad a view of the optimizer's flat gradient buffer
# (optimus/optimizers.py:105-111), zeroed in place (:117-118) and accumulated into over the
# micro-batches of a step (dist_train.py:154), so autograd finishes each weight-gradient GEMM with an
# elementwise `p.grad += dW` over the whole weight.  When a weight's .grad is such a live view the
# backward functions below let the GEMM's epilogue do that sum (the *_accumulate entry points: the
# same bits) and hand autograd None for the weight.  Set to False to always return fresh gradients.
accumulate_weight_grads_in_place = True


def _live_grad(param):
    """param.grad if the weight-gradient kernels may add into it in place: a leaf parameter whose
    gradient already exists as a dense view of a larger buffer, same dtype and shape, with no hooks
    that would have to see the incoming gradient; else None."""
    if not accumulate_weight_grads_in_place or torch.is_grad_enabled():
        return None                     # (grad mode is on in backward only under create_graph)
    return _n.host().live_grad(param)


# ----------------------------------------------------------------------------------------------
# Grouped GEMM functions
# ----------------------------------------------------------------------------------------------
class GroupedGemmFunction(torch.autograd.Function):
    """out[s:e] = in[s:e] @ W[g].T per expert segment (reference moe.py:163-215).

    `max_tokens_per_expert` and `use_triton_path` exist for signature parity and are ignored:
    the kernel sizes its grid from the row count and reads the offsets on the device."""

    @staticmethod
    def forward(ctx, input, merged_weight, cum_token_counts, max_tokens_per_expert=None,
                use_triton_path=False):
        _gemm_dtype(input, merged_weight)
        _n.require_cuda_contiguous(input)
        num_tokens = input.shape[0]
        num_experts, ofm, ifm = merged_weight.shape
        cum = _device_counts(cum_token_counts, input.device)
        output = torch.empty((num_tokens, ofm), dtype=input.dtype, device=input.device)
        _grouped_gemm("fwd", input, merged_weight, output, cum, num_tokens, num_experts, ofm, ifm,
                      _expert_stride(merged_weight))
        ctx.save_for_backward(input, merged_weight, cum)
        return output

    @staticmethod
    def backward(ctx, output_grad):
        input, merged_weight, cum = ctx.saved_tensors
        output_grad = output_grad.contiguous()
        num_experts, ofm, ifm = merged_weight.shape
        rows = input.shape[0]
        input_grad = torch.empty_like(input)
        weight_grad = _live_grad(merged_weight)
        acc = weight_grad is not None
        if not acc:
            weight_grad = torch.empty((num_experts, ofm, ifm), dtype=merged_weight.dtype, device=merged_weight.device)
        pitch = _expert_stride(weight_grad)
        _grouped_gemm("dgrad", output_grad, merged_weight, input_grad, cum, rows, num_experts, ofm, ifm,
                      _expert_stride(merged_weight))
        _grouped_gemm("wgrad", output_grad, input, weight_grad, cum, rows, num_experts, ofm, ifm, pitch,
                      accumulate=acc)
        return input_grad, (None if acc else weight_grad), None, None, None


def _expert_views(weight_tuple):
    """[gate, up, down] as [G, out, in] views over the per-expert matrices of a (gate_0, up_0, down_0,
    gate_1, ...) tuple, which must lie at a constant pitch in one buffer."""
    return [_n.host().expert_view(list(weight_tuple[j::3])) for j in range(3)]


class MergedMLPFunction(torch.autograd.Function):
    """y = (silu(x Wg^T) * (x Wu^T)) Wd^T per expert segment, with the fused kernels:
    gate+up+SwiGLU in one launch forward; backward = down dgrad fused with the SwiGLU backward,
    one dual-operand dgrad for dx, and three weight-gradient GEMMs (in one launch where that is sooner; float32: in one
    launch with the dgrad).

    Same mathematics as the three GroupedGemmFunction calls and two elementwise ops of the
    reference's MergedMLP.forward (moe.py:396-405) under autograd; g and u are kept in the module's
    dtype for the backward like the reference keeps output_gproj / output_uproj."""

    @staticmethod
    def forward(ctx, x, w_gate, w_up, w_down, cum_token_counts):
        # a single MLP may hand its three [out, in] weights over as they are
        ctx.leaves = [w_gate, w_up, w_down]
        y, *state = _n.host().merged_mlp_forward(x, cum_token_counts, ctx.leaves, None)
        ctx.save_for_backward(x, *state, *ctx.leaves)
        return y

    @staticmethod
    def backward(ctx, dy):
        *saved, w_gate, w_up, w_down = ctx.saved_tensors
        return (*_n.host().merged_mlp_backward(dy, *saved, [w_gate, w_up, w_down], ctx.leaves, True, None, None, None),
                None)


class GatheredMergedMLPFunction(torch.autograd.Function):
    """PrepareInputForGroupGemmFunction followed by MergedMLPFunction (reference moe.py:217-282 and
    :396-405) without the gathered copy of the activations: the gate/up forward GEMM and the two
    gate/up weight-gradient GEMMs read hidden_states through input_indices.  Bit-identical to the
    two functions in sequence; backward ends with the same per-token reduction of the routed rows'
    gradients (shuffle_sub_matrix_reduce)."""

    @staticmethod
    def forward(ctx, hidden_states, input_indices, cum_expert_counts_ep, output_indices, w_gate, w_up, w_down,
                cum_token_counts):
        hidden_states = hidden_states.contiguous()
        ctx.leaves = [w_gate, w_up, w_down]
        y, *state = _n.host().merged_mlp_forward(hidden_states, cum_token_counts, ctx.leaves, input_indices)
        ctx.save_for_backward(input_indices, cum_expert_counts_ep, output_indices, hidden_states, *state, *ctx.leaves)
        return y

    @staticmethod
    def backward(ctx, dy):
        *saved, w_gate, w_up, w_down = ctx.saved_tensors
        dx, *dws = _n.host().merged_mlp_backward(dy, *saved[3:], [w_gate, w_up, w_down], ctx.leaves, True, *saved[:3])
        return (dx, None, None, None, *dws, None)


class GroupMLPFunction(torch.autograd.Function):
    """Un-merged layout of the reference (moe.py:43-161): weights arrive as 3*N separate
    [out, in] tensors (gate_0, up_0, down_0, gate_1, ...).  They must sit at one constant pitch
    inside a single buffer (true for parameters re-pointed into MixedPrecisionAdamW.flat_param and
    after pack_expert_weights); the same fused kernels then run on strided views, no copies."""

    @staticmethod
    def forward(ctx, input, cum_token_counts, use_triton_path, *weight_tuple):
        ctx.leaves = list(weight_tuple)
        views = _expert_views(weight_tuple)
        y, *state = _n.host().merged_mlp_forward(input, cum_token_counts, views, None)
        ctx.save_for_backward(input, *state, *views)
        return y

    @staticmethod
    def backward(ctx, output_grad):
        *saved, wg, wu, wd = ctx.saved_tensors
        dx, *dws = _n.host().merged_mlp_backward(output_grad, *saved, [wg, wu, wd], ctx.leaves, False, None, None, None)
        return (dx, None, None, *dws)


class GatheredGroupMLPFunction(torch.autograd.Function):
    """GroupMLPFunction on hidden_states[input_indices] without the gathered copy (see
    GatheredMergedMLPFunction); weights as in GroupMLPFunction."""

    @staticmethod
    def forward(ctx, hidden_states, input_indices, cum_expert_counts_ep, output_indices, cum_token_counts,
                *weight_tuple):
        hidden_states = hidden_states.contiguous()
        ctx.leaves = list(weight_tuple)
        views = _expert_views(weight_tuple)
        y, *state = _n.host().merged_mlp_forward(hidden_states, cum_token_counts, views, input_indices)
        ctx.save_for_backward(input_indices, cum_expert_counts_ep, output_indices, hidden_states, *state, *views)
        return y

    @staticmethod
    def backward(ctx, output_grad):
        *saved, wg, wu, wd = ctx.saved_tensors
        dx, *dws = _n.host().merged_mlp_backward(output_grad, *saved[3:], [wg, wu, wd], ctx.leaves, False, *saved[:3])
        return (dx, None, None, None, None, *dws)


def routed_mlp_unfit_reason(hidden_states, routing_weights, w_gate, w_down):
    """None when RoutedMLPFunction's kernels take these operands (bf16 activations and expert
    weights on the GPU, fp32 or bf16 routing weights, H and I multiples of 8), else why not."""
    I, H = w_gate.shape[-2:]
    if not (hidden_states.is_cuda and hidden_states.dim() == 2):
        return "the hidden states are not a 2-D device tensor"
    if not (hidden_states.dtype == torch.bfloat16 and w_gate.dtype == torch.bfloat16
            and w_down.dtype == torch.bfloat16):
        return f"activations / expert weights are not bfloat16 ({hidden_states.dtype}, {w_gate.dtype})"
    if routing_weights.dtype not in (torch.bfloat16, torch.float32):
        return f"routing weights are {routing_weights.dtype}"
    if H % 8 != 0 or I % 8 != 0:
        return f"hidden size {H} / ffn size {I} are not multiples of 8"
    return None


def routed_mlp_kernel_fits(hidden_states, routing_weights, w_gate, w_down):
    """True when RoutedMLPFunction's kernels take these operands."""
    return routed_mlp_unfit_reason(hidden_states, routing_weights, w_gate, w_down) is None


class RoutedMLPFunction(torch.autograd.Function):
    """The expert half of the block in one function: PrepareInputForGroupGemmFunction, the SwiGLU
    MLP of every expert and GroupGemmOutputReductionFunction (reference moe.py:217-405), with both
    row permutations and the routing weight folded into the GEMMs:

      forward   h = w[t,k] * silu(x Wg^T) * (x Wu^T) formed in the gate+up epilogue (x read through
                input_indices), y = h Wd^T, final[t] = (residual[t] +) sum of the token's rows of y;
      backward  the down projection's two backward GEMMs read dfinal through input_indices, the
                SwiGLU-backward epilogue applies w and forms the routing weights' gradient
                sum_i (dfinal Wd)[i] * silu(g)[i] * u[i]; the rest as GatheredMergedMLPFunction.

    Neither the gathered input, nor the experts' output gradient w[t,k] * dfinal[t] (both [rows, H])
    is written.  The weight commutes with the linear down projection, so this is the reference's
    mathematics; h is rounded to bf16 after the weight instead of before, so results agree with the
    separate functions to bf16 accuracy, not bit for bit.

    `weights`: (gate, up, down) as [G, I, H] / [G, H, I] tensors when n_merged is true, else the
    3*G per-expert matrices of GroupMLPFunction."""

    @staticmethod
    def forward(ctx, hidden_states, routing_weights, input_indices, cum_expert_counts_ep, output_indices,
                selected_experts_indices, cum_token_counts, residual, n_merged, *weights):
        # n_merged: True = merged weights; False = per-expert weights; "bound" forms of both say that
        # the index arrays are sized by an upper bound of the routed rows (expert_computation)
        ctx.rows_is_bound = n_merged in ("merged_bound", "per_expert_bound")
        ctx.n_merged = n_merged in (True, "merged_bound")
        ctx.has_residual = residual is not None
        ctx.leaves = list(weights)
        views = ctx.leaves if ctx.n_merged else _expert_views(weights)
        index = (input_indices, cum_expert_counts_ep, output_indices, selected_experts_indices)
        hidden_states, routing_weights = hidden_states.contiguous(), routing_weights.contiguous()
        final, *state = _n.host().routed_mlp_forward(hidden_states, routing_weights, *index, cum_token_counts, residual,
                                                     views)
        ctx.save_for_backward(hidden_states, routing_weights, *index, *state, *views)
        return final

    @staticmethod
    def backward(ctx, dfinal):
        *saved, wg, wu, wd = ctx.saved_tensors
        dx, drw, *dws = _n.host().routed_mlp_backward(dfinal, *saved, [wg, wu, wd], ctx.leaves, ctx.n_merged,
                                                      ctx.rows_is_bound, None)
        return (dx, drw, None, None, None, None, None, dfinal if ctx.has_residual else None, None, *dws)


class RoutedAndSharedMLPFunction(torch.autograd.Function):
    """shared_mlp(x) + the routed experts' weighted sum (reference modeling_deepseek_v3.py:265,
    `self.moe(...) + self.shared_experts(residuals)`) as one function: RoutedMLPFunction over the
    per-expert weights with the shared MLP's output as its residual.  Same kernels and bits forward
    as the two functions in sequence.  Backward runs the shared MLP first and hands its input
    gradient to the routed experts' per-token sum as the base it adds to, so the two input
    gradients meet inside a kernel (base + cast(sum): what autograd's accumulation gives) and no
    separate [T,H] addition runs.

    weights: the 3*G routed matrices in GroupMLPFunction's order, then the shared MLP's gate, up,
    down [out, in] matrices."""

    @staticmethod
    def forward(ctx, hidden_states, routing_weights, input_indices, cum_expert_counts_ep, output_indices,
                selected_experts_indices, cum_token_counts, rows_is_bound, *weights):
        ctx.leaves, ctx.shared_leaves = list(weights[:-3]), list(weights[-3:])
        ctx.rows_is_bound = bool(rows_is_bound)
        views = _expert_views(ctx.leaves)
        index = (input_indices, cum_expert_counts_ep, output_indices, selected_experts_indices)
        hidden_states, routing_weights = hidden_states.contiguous(), routing_weights.contiguous()
        one = single_segment_counts(hidden_states.shape[0], hidden_states.device)
        y_shared, *shared_state = _n.host().merged_mlp_forward(hidden_states, one, ctx.shared_leaves, None)
        final, *state = _n.host().routed_mlp_forward(hidden_states, routing_weights, *index, cum_token_counts, y_shared,
                                                     views)
        ctx.save_for_backward(hidden_states, routing_weights, *index, *state, *views, *shared_state, *ctx.shared_leaves)
        return final

    @staticmethod
    def backward(ctx, dfinal):
        saved = ctx.saved_tensors
        routed, views, shared_state, shared = saved[:11], saved[11:14], saved[14:18], saved[18:]
        # first the shared MLP: its input gradient is the base of the routed experts' per-token sum
        base, *dws_shared = _n.host().merged_mlp_backward(dfinal, routed[0], *shared_state, list(shared), ctx.shared_leaves,
                                                          True, None, None, None)
        dx, drw, *dws = _n.host().routed_mlp_backward(dfinal, *routed, list(views), ctx.leaves, False, ctx.rows_is_bound,
                                                      base)
        return (dx, drw, None, None, None, None, None, None, *dws, *dws_shared)


def has_constant_pitch(weights):
    """True when the matrices lie at one constant pitch inside one buffer."""
    return _n.host().constant_pitch(list(weights))


def pack_expert_weights(experts, names=("gate_proj", "up_proj", "down_proj")):
    """Make the [out, in] weights of a ModuleList of expert MLPs lie at a constant pitch: where
    they do not already, re-point them into one buffer per projection (p.data becomes a view,
    values kept).  Module.to()/.bfloat16() re-allocates parameters one by one, so the blocks call
    this before they hand the weights to the grouped kernels."""
    for name in names:
        ws = [getattr(e, name).weight for e in experts]
        if has_constant_pitch([w.data for w in ws]):
            continue
        buf = torch.stack([w.data for w in ws]).contiguous()
        for n, w in enumerate(ws):
            w.data = buf[n]


def packed_expert_parameters(experts):
    """The (gate, up, down) weights of every expert in GroupMLPFunction's order, packed (see
    pack_expert_weights)."""
    params = _n.host().expert_parameters(experts)
    if not all(_n.host().constant_pitch(params[j::3]) for j in range(3)):
        pack_expert_weights(experts)
        params = _n.host().expert_parameters(experts)
    return params


def group_mlp(x, cum_token_counts, experts, input_indices=None, cum_expert_counts_ep=None, output_indices=None):
    """The expert MLPs of a ModuleList on x (GroupMLPFunction), or on x[input_indices] (GatheredGroupMLPFunction)."""
    return _n.host().merged_mlp(x, cum_token_counts, False, packed_expert_parameters(experts), input_indices,
                                cum_expert_counts_ep, output_indices)


class PrepareInputForGroupGemmFunction(torch.autograd.Function):
    """K4: ggemm_input = hidden_states[input_indices]; backward sums each token's routed rows in
    fp32 (reference moe.py:217-282).  The four trailing flags are accepted and ignored."""

    @staticmethod
    def forward(ctx, hidden_states, input_indices, cum_expert_counts_ep, output_indices,
                use_ref_path_fwd=False, use_ref_path_bwd=False,
                use_triton_path_fwd=False, use_triton_path_bwd=False):
        num_tokens, hidden_dim = hidden_states.shape
        num_routed_tokens = input_indices.shape[0]
        with record_pcl_function("1moeblock--6gmlp_input_prep_fwd"):
            ggemm_input = torch.empty((num_routed_tokens, hidden_dim), dtype=hidden_states.dtype,
                                      device=hidden_states.device)
            pcl_xpu_customops.index_gather(hidden_states.contiguous(), input_indices, ggemm_input)
        ctx.save_for_backward(cum_expert_counts_ep, output_indices)
        ctx.num_tokens = num_tokens
        ctx.hidden_dim = hidden_dim
        return ggemm_input

    @staticmethod
    def backward(ctx, ggemm_input_grad):
        cum_expert_counts_ep, output_indices = ctx.saved_tensors
        with record_pcl_function("1moeblock--6gmlp_input_prep_bwd"):
            ggemm_input_grad = ggemm_input_grad.contiguous()
            hidden_states_grad = torch.empty((ctx.num_tokens, ctx.hidden_dim),
                                             dtype=ggemm_input_grad.dtype,
                                             device=ggemm_input_grad.device)
            pcl_xpu_customops.shuffle_sub_matrix_reduce(ggemm_input_grad, cum_expert_counts_ep,
                                                        output_indices, hidden_states_grad)
        return hidden_states_grad, None, None, None, None, None, None, None


class GroupGemmOutputReductionFunction(torch.autograd.Function):
    """K6: final[t] = sum_k w[t,k] * ggemm_output[pos(t,k)] in fp32, one rounding; backward gives
    ggemm_output_grad and routing_weights_grad (reference moe.py:284-377).  The four trailing
    flags are accepted and ignored.  routing_weights may be fp32 while activations are bf16."""

    @staticmethod
    def forward(ctx, ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices,
                input_indices, output_indices,
                use_ref_path_fwd=False, use_ref_path_bwd=False,
                use_triton_path_fwd=False, use_triton_path_bwd=False):
        return _combine_forward(ctx, ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices,
                                input_indices, output_indices, None)

    @staticmethod
    def backward(ctx, final_hidden_states_grad):
        return (*_n.host().combine_backward(final_hidden_states_grad, *ctx.saved_tensors), *(None,) * 8)


class GroupGemmOutputReductionResidualFunction(torch.autograd.Function):
    """residual + GroupGemmOutputReductionFunction(...) in one pass: the combined sum is rounded to
    the activation dtype and then added to `residual` (both roundings of the two-step form).  Used
    for the decoder layer's residual connection (modeling_olmoe.py:415) and for the DeepSeek-V3
    block's routed + shared sum (modeling_deepseek_v3.py:265).  The gradient of the output goes to
    `residual` unchanged and into the combine's backward."""

    @staticmethod
    def forward(ctx, ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices,
                input_indices, output_indices, residual):
        return _combine_forward(ctx, ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices,
                                input_indices, output_indices, residual)

    @staticmethod
    def backward(ctx, final_hidden_states_grad):
        return (*_n.host().combine_backward(final_hidden_states_grad, *ctx.saved_tensors), None, None, None, None,
                final_hidden_states_grad)


def _combine_forward(ctx, ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices, input_indices,
                     output_indices, residual):
    routing_weights = routing_weights.contiguous()
    ctx.save_for_backward(ggemm_output, routing_weights, selected_experts_indices, input_indices, output_indices)
    return _n.host().combine(ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices, input_indices,
                             output_indices, residual)


# ----------------------------------------------------------------------------------------------
# Modules
# ----------------------------------------------------------------------------------------------
class MergedMLP(nn.Module):
    """All local experts' SwiGLU MLPs as three 3-D parameters (reference moe.py:379-405)."""

    def __init__(self, config):
        super(MergedMLP, self).__init__()
        self.config = config
        self.num_experts_per_rank = config.num_experts // config.expert_parallelism
        self.gate_proj_merged_weight = torch.nn.Parameter(
            torch.empty((self.num_experts_per_rank, config.intermediate_size, config.hidden_size)))
        self.up_proj_merged_weight = torch.nn.Parameter(
            torch.empty((self.num_experts_per_rank, config.intermediate_size, config.hidden_size)))
        self.down_proj_merged_weight = torch.nn.Parameter(
            torch.empty((self.num_experts_per_rank, config.hidden_size, config.intermediate_size)))

    def _weights(self):
        return [self.gate_proj_merged_weight, self.up_proj_merged_weight, self.down_proj_merged_weight]

    def forward(self, input, cum_token_counts):
        return _n.host().merged_mlp(input, cum_token_counts, True, self._weights(), None, None, None)

    def forward_gathered(self, hidden_states, input_indices, cum_expert_counts_ep, output_indices,
                         cum_token_counts):
        """forward(hidden_states[input_indices], cum_token_counts) with the gather folded into the
        GEMMs; the two index arrays after input_indices serve the backward's per-token reduction."""
        return _n.host().merged_mlp(hidden_states, cum_token_counts, True, self._weights(), input_indices,
                                    cum_expert_counts_ep, output_indices)


def expert_computation(hidden_states, routing_weights, selected_experts, expert_start_idx,
                       expert_end_idx, experts_fn, num_total_experts, gathered_experts_fn=None,
                       residual=None, routed_experts_fn=None, sync_free_window=False, fused_experts_fn=None):
    """K1..K6 for 2-D hidden_states [T,H]: permute, run `experts_fn(ggemm_input, cum_token_counts)`,
    combine.  Shared by the OLMoE and DeepSeek-V3 blocks.  With `gathered_experts_fn(hidden_states,
    input_indices, cum_expert_counts_ep, output_indices, cum_token_counts)` the experts read the
    tokens through the index and K4's gathered copy is not built.  With `residual` [T,H] the result
    is residual + combine(...), added inside the combine kernel.  `routed_experts_fn(hidden_states,
    routing_weights, input_indices, cum_expert_counts_ep, output_indices, selected_experts_indices,
    cum_token_counts, residual)` may do gather, experts and combine in one function
    (RoutedMLPFunction); it returns None when its kernels do not take the operands.
    `fused_experts_fn(hidden_states, routing_weights, selected_experts, residual)` does the same
    including the permutation, whose arrays then never become Python objects: what the blocks pass
    (moe_experts of the host module); `routed_experts_fn` serves callers with an expert function of
    their own.

    Under an expert window the number of routed rows is only known on the device.  It is read back
    once, like the reference does (moe.py:520), by the fused function only where activations for all
    T*K pairs would take too much memory (sized_by_bound).  With `sync_free_window` and a
    `routed_experts_fn`, or a block's `sync_free_expert_window`, nothing is ever read back: the index
    arrays keep their T*K entries (om_moe_sort marks the unused tail), the activations of the expert
    MLP are allocated for T*K rows, of which only the routed ones are computed, and the function is
    called with `rows_is_bound=True`.  That makes the step capturable in a HIP graph at the price of
    expert_parallelism times the activation memory."""
    if fused_experts_fn is not None:
        final = fused_experts_fn(hidden_states, routing_weights, selected_experts, residual)
        if final is not None:
            return final
    T, K = selected_experts.shape
    with record_pcl_function("1moeblock--3index_calculation"):
        (cum_token_counts, cum_expert_counts_ep, input_indices, output_indices,
         selected_experts_indices) = build_token_permutation(selected_experts, expert_start_idx,
                                                             expert_end_idx)
    windowed = not (expert_start_idx == 0 and expert_end_idx == num_total_experts)
    if windowed and sync_free_window and routed_experts_fn is not None:
        final = routed_experts_fn(hidden_states, routing_weights, input_indices, cum_expert_counts_ep,
                                  output_indices, selected_experts_indices, cum_token_counts, residual,
                                  rows_is_bound=True)
        if final is not None:
            return final
    if not windowed:
        num_routed_tokens = T * K            # every pair is local: no host read
    else:
        num_routed_tokens = int(cum_token_counts[-1].item())   # same host read as moe.py:520
    input_indices = input_indices[:num_routed_tokens]
    output_indices = output_indices[:num_routed_tokens]
    selected_experts_indices = selected_experts_indices[:num_routed_tokens]
    if routed_experts_fn is not None:
        final = routed_experts_fn(hidden_states, routing_weights, input_indices, cum_expert_counts_ep,
                                  output_indices, selected_experts_indices, cum_token_counts, residual)
        if final is not None:
            return final
    if gathered_experts_fn is not None:
        ggemm_output = gathered_experts_fn(hidden_states, input_indices, cum_expert_counts_ep,
                                           output_indices, cum_token_counts)
    else:
        ggemm_input = PrepareInputForGroupGemmFunction.apply(hidden_states, input_indices,
                                                             cum_expert_counts_ep, output_indices)
        ggemm_output = experts_fn(ggemm_input, cum_token_counts)
    return _n.host().combine(ggemm_output, routing_weights, cum_expert_counts_ep, selected_experts_indices,
                             input_indices, output_indices, residual)


class FastOlmoeParallelSparseMoeBlock(nn.Module):
    """Reference moe.py:407-632.  forward(hidden_states [B,S,H]) ->
    (final_hidden_states [B,S,H], router_logits [B*S,N] or None).

    Limits of a bfloat16 block (a shape outside them raises, nothing falls back to a library):
    at most 256 experts in the gate; hidden size and ffn size multiples of 8."""

    def __init__(self, config, pmap=None):
        super().__init__()
        from optimus.models.olmoe.modeling_olmoe import OlmoeParallelMLP
        self.config = config
        self.pmap = pmap
        self.num_experts_per_rank = config.num_experts // config.expert_parallelism
        self.expert_start_idx = self.pmap.ep_ind * self.num_experts_per_rank
        self.expert_end_idx = (self.pmap.ep_ind + 1) * self.num_experts_per_rank

        self.hidden_size = config.hidden_size
        self.intermediate_size = config.intermediate_size
        self.num_experts = config.num_experts
        self.num_experts_per_tok = config.num_experts_per_tok
        self.norm_topk_prob = config.norm_topk_prob
        self.output_router_logits = config.output_router_logits

        self.gate = nn.Linear(self.hidden_size, self.num_experts, bias=False)
        if not self.config.use_merged_mlp_in_fast_moe:
            self.experts = nn.ModuleList([OlmoeParallelMLP(config) for _ in range(self.num_experts_per_rank)])
        else:
            self.experts = MergedMLP(config)

        self.use_activation_checkpointing_for_moe = False
        if config.use_activation_checkpointing:
            self.use_activation_checkpointing_for_moe = config.activation_checkpointing_level & (1 << 0)

        if getattr(config, "force_uniform_routing", False):
            raise NotImplementedError("force_uniform_routing is a debug mask of the reference "
                                      "(moe.py:459-464) and is not part of this build")
        # fp32 router logits (x.float() @ Wg.float().T) instead of model-dtype logits
        self.router_logits_fp32 = bool(getattr(config, "router_logits_fp32", False))
        # merged experts read the tokens through input_indices instead of a gathered copy
        self.fuse_input_gather = bool(getattr(config, "fuse_input_gather", True))
        # the routing weight is applied inside the expert MLP and the combine's backward is folded
        # into the down projection's backward GEMMs (RoutedMLPFunction); needs fuse_input_gather
        self.fuse_routing_weights = bool(getattr(config, "fuse_routing_weights", True))
        # under an expert window: never read the routed row count back (see expert_computation)
        self.sync_free_expert_window = bool(getattr(config, "sync_free_expert_window", False))

    def _experts_fn(self, ggemm_input, cum_token_counts):
        if isinstance(self.experts, MergedMLP):
            return self.experts(ggemm_input, cum_token_counts)
        return group_mlp(ggemm_input, cum_token_counts, self.experts)

    def _gathered_experts_fn(self, hidden_states, input_indices, cum_expert_counts_ep, output_indices,
                             cum_token_counts):
        if isinstance(self.experts, MergedMLP):
            return self.experts.forward_gathered(hidden_states, input_indices, cum_expert_counts_ep,
                                                 output_indices, cum_token_counts)
        return group_mlp(hidden_states, cum_token_counts, self.experts, input_indices, cum_expert_counts_ep,
                         output_indices)

    def _fused_experts_fn(self, hidden_states, routing_weights, selected_experts, residual, sorted_index=None):
        """Permutation and RoutedMLPFunction in one call; None when the kernels do not take the operands.
        `sorted_index`: the permutation, where the router's launch has made it."""
        merged = isinstance(self.experts, MergedMLP)
        if merged:
            # (as attributes: a weight may be parametrized, or a plain tensor that a wrapper has put there)
            weights = self.experts._weights()
        else:
            weights = packed_expert_parameters(self.experts)
        why = routed_mlp_unfit_reason(hidden_states, routing_weights, weights[0], weights[2])
        if why is not None:
            if hidden_states.dtype == torch.bfloat16:    # (float32 modules apply the weight in the combine, by design)
                note_unfused_path("routing weight inside the expert MLP", why)
            return None
        return _n.host().moe_experts(hidden_states, routing_weights, selected_experts, self.expert_start_idx,
                                     self.expert_end_idx, self.num_experts, self.sync_free_expert_window,
                                     residual, merged, weights, False, None, sorted_index)

    def forward_with_residual(self, hidden_states, residual):
        """(residual + forward(hidden_states)[0], router_logits): the decoder layer's
        `hidden_states = residual + hidden_states` after the block (modeling_olmoe.py:415) folded into
        the combine kernel; same bits as the two steps."""
        return self.forward(hidden_states, residual=residual)

    def forward(self, hidden_states, residual=None):
        batch_size, sequence_length, hidden_dim = hidden_states.shape
        flat = hidden_states.reshape(-1, hidden_dim)
        gate_unfit = gate_kernel_unfit_reason(flat, self.gate.weight) if self.router_logits_fp32 else None
        if self.router_logits_fp32 and gate_unfit is not None and flat.dtype == torch.bfloat16:
            note_unfused_path("gate projection fused with the routing", gate_unfit,
                              instead="running the kernels of other hidden sizes (same fp32 logits): one launch for a small gate, "
                                      "else the projection and the routing as separate kernels")
        # (the experts are fed from the router's pass-through of the hidden states, so that their input
        # gradient and the gate's are added in one kernel)
        weight = self.gate.weight.contiguous()
        sorted_index = None
        if flat.is_cuda and flat.dtype == weight.dtype and flat.dtype in (torch.bfloat16, torch.float32) \
                and self.gate.bias is None:
            bf16 = flat.dtype == torch.bfloat16
            # (the router sorts its selections where one launch can, for the experts called right behind it)
            sorts = bf16 and self.fuse_input_gather and self.fuse_routing_weights and not self.use_activation_checkpointing_for_moe
            routing_weights, selected_experts, router_logits, flat, sorted_index = _n.host().route_softmax_sorted(
                flat.contiguous(), weight, self.num_experts_per_tok, bool(self.norm_topk_prob), flat.dtype,
                self.router_logits_fp32 and gate_unfit is None, bf16 and not self.router_logits_fp32,
                self.expert_start_idx if sorts else 0, self.expert_end_idx if sorts else 0)
        else:
            if self.router_logits_fp32:
                router_logits, flat = fp32_logits_with_passthrough(flat, weight)
            else:
                router_logits, flat = gate_logits_with_passthrough(flat, self.gate)
            routing_weights, selected_experts = SoftmaxTopkRouterFunction.apply(
                router_logits.contiguous(), self.num_experts_per_tok, self.norm_topk_prob, flat.dtype)

        def expert_computation_block(flat, selected_experts, routing_weights, residual=None):
            gathered = self._gathered_experts_fn if self.fuse_input_gather else None
            fused = self._fused_experts_fn if (self.fuse_input_gather and self.fuse_routing_weights) else None
            if sorted_index is not None:
                fused = functools.partial(fused, sorted_index=sorted_index)
            return expert_computation(flat, routing_weights, selected_experts,
                                      self.expert_start_idx, self.expert_end_idx, self._experts_fn,
                                      self.num_experts, gathered_experts_fn=gathered,
                                      residual=None if residual is None else residual.reshape(-1, hidden_dim),
                                      fused_experts_fn=fused)

        args = [flat, selected_experts, routing_weights]
        if residual is not None:
            args.append(residual)
        if self.use_activation_checkpointing_for_moe:
            final_hidden_states = torch_activation_checkpoint(expert_computation_block, *args,
                                                              use_reentrant=False)
        else:
            final_hidden_states = expert_computation_block(*args)
        final_hidden_states = final_hidden_states.reshape(batch_size, sequence_length, hidden_dim)

        if self.output_router_logits:
            return final_hidden_states, router_logits
        return final_hidden_states, None

    def set_parameters_from_full_module(self, module):
        self.gate.load_state_dict(module.gate.state_dict())
        with torch.no_grad():
            for local_expert_idx in range(self.num_experts_per_rank):
                src = module.experts[self.expert_start_idx + local_expert_idx]
                if isinstance(self.experts, MergedMLP):
                    self.experts.gate_proj_merged_weight[local_expert_idx].copy_(src.gate_proj.weight.data)
                    self.experts.up_proj_merged_weight[local_expert_idx].copy_(src.up_proj.weight.data)
                    self.experts.down_proj_merged_weight[local_expert_idx].copy_(src.down_proj.weight.data)
                else:
                    self.experts[local_expert_idx].load_state_dict(src.state_dict())


# ----------------------------------------------------------------------------------------------
# Checkpoint interchange between the merged and the per-expert weight layouts
# ----------------------------------------------------------------------------------------------
_MERGED_SUFFIX = "_merged_weight"


def merged_state_dict_to_per_expert(state_dict, expert_start_id=0):
    """Rewrites '<p>.experts.<lin>_merged_weight' [NR,out,in] entries as NR entries
    '<p>.experts.<id>.<lin>.weight' (views, no copies), id = expert_start_id + local index; all
    other entries pass through.  This is the un-merging the reference does when it converts an
    expert-parallel rank's checkpoint to per-expert keys
    (evals/convert_olmoe_om_checkpoint_to_hf.py:59-88)."""
    out = {}
    for name, tensor in state_dict.items():
        tokens = name.split(".")
        if "experts" in tokens and tokens[-1].endswith(_MERGED_SUFFIX):
            linear_key = tokens[-1][: -len(_MERGED_SUFFIX)]
            for local in range(tensor.shape[0]):
                serial = ".".join(tokens[:-1] + [str(expert_start_id + local), linear_key, "weight"])
                out[serial] = tensor[local]
        else:
            out[name] = tensor
    return out


def per_expert_state_dict_to_merged(state_dict, num_local_experts, expert_start_id=0):
    """The inverse: gathers '<p>.experts.<id>.<lin>.weight' for id in
    [expert_start_id, expert_start_id + num_local_experts) into '<p>.experts.<lin>_merged_weight'
    (one stacked tensor per projection); entries of experts outside the window are dropped, all
    other entries pass through.  Same mapping as the reference's checkpoint generator for
    use_merged_mlp_in_fast_moe (generate_parallel_model.py:136-148)."""
    out, groups = {}, {}
    for name, tensor in state_dict.items():
        tokens = name.split(".")
        if "experts" in tokens:
            i = tokens.index("experts")
            if len(tokens) == i + 4 and tokens[i + 1].isdigit() and tokens[-1] == "weight":
                local = int(tokens[i + 1]) - expert_start_id
                if 0 <= local < num_local_experts:
                    key = ".".join(tokens[: i + 1] + [tokens[i + 2] + _MERGED_SUFFIX])
                    groups.setdefault(key, {})[local] = tensor
                continue
        out[name] = tensor
    for key, parts in groups.items():
        missing = [expert_start_id + j for j in range(num_local_experts) if j not in parts]
        if missing:
            raise KeyError(f"{key}: no weights for experts {missing}")
        out[key] = torch.stack([parts[j] for j in range(num_local_experts)])
    return out

