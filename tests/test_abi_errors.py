"""Error convention of the C ABI: every entry point validates its arguments before it touches the
HIP runtime and answers with a negative OM_ERR_* code — it never throws and never launches on bad
input.  These calls return from the validation, so they run without a GPU; the pointers are made-up
addresses that are never dereferenced on the host."""
import ctypes
import struct

import pytest

from optimus import _native as n

OK, NULL, DTYPE, SHAPE, ALIGN, LAUNCH, WORKSPACE = 0, -1, -2, -3, -4, -5, -6
P = 0x7f0000001000        # a 16-byte aligned, never dereferenced "device pointer"
ODD = P + 8               # misaligned
BF16, F32, I64 = n.OM_BF16, n.OM_F32, 1


@pytest.fixture(scope="module")
def lib():
    return n.lib()


def test_strerror_names_every_code(lib):
    texts = {c: lib.om_strerror(c).decode() for c in (OK, NULL, DTYPE, SHAPE, ALIGN, LAUNCH, WORKSPACE)}
    assert len(set(texts.values())) == 7 and all(texts.values())
    assert "unknown" in lib.om_strerror(-99).decode()


def test_adamw(lib):
    hp = (4e-4, 0.9, 0.95, 1e-8, 0.1)
    assert lib.om_adamw_step(P, P, P, P, P, 16, *hp, 1, 7, None) == DTYPE
    assert lib.om_adamw_step(P, P, P, P, P, 16, *hp, 0, BF16, None) == SHAPE      # step is 1-based
    assert lib.om_adamw_step(P, P, P, P, P, -1, *hp, 1, BF16, None) == SHAPE
    assert lib.om_adamw_step(P, P, P, P, P, 0, *hp, 1, BF16, None) == OK          # nothing to do
    assert lib.om_adamw_step(P, None, P, P, P, 16, *hp, 1, BF16, None) == NULL
    assert lib.om_adamw_step(None, P, P, P, P, 16, *hp, 1, BF16, None) == NULL    # bf16 mode needs param
    assert lib.om_adamw_step(P, P, ODD, P, P, 16, *hp, 1, BF16, None) == ALIGN
    assert lib.om_adamw_step_clipped(P, P, P, P, P, 16, *hp, 1, BF16, None, 1, None) == NULL   # no scale
    assert lib.om_adamw_step_clipped(P, P, P, P, P, 16, *hp, 1, 9, P, 1, None) == DTYPE


def test_grad_norm(lib):
    assert lib.om_grad_sumsq(P, 5, P, 4, P, None) == DTYPE
    assert lib.om_grad_sumsq(P, BF16, P, -1, P, None) == SHAPE
    assert lib.om_grad_sumsq(P, BF16, P, 0, P, None) == OK
    assert lib.om_grad_sumsq(None, BF16, P, 4, P, None) == NULL
    assert lib.om_grad_sumsq(ODD, BF16, P, 4, P, None) == ALIGN
    assert lib.om_grad_norm_clip_coef(P, P, 0, BF16, 1.0, P, P, P, None) == SHAPE
    assert lib.om_grad_norm_clip_coef(P, P, 3, BF16, 1.0, None, P, P, None) == NULL
    assert lib.om_grad_norm_clip_coef(P, P, 3, 4, 1.0, P, P, P, None) == DTYPE


def test_routers(lib):
    assert lib.om_route_softmax_topk(P, 3, 8, 64, 8, 0, P, BF16, P, None) == DTYPE
    assert lib.om_route_softmax_topk(P, F32, 8, 600, 8, 0, P, BF16, P, None) == SHAPE      # N > 512
    assert lib.om_route_softmax_topk(P, F32, 8, 4, 8, 0, P, BF16, P, None) == SHAPE        # K > N
    assert lib.om_route_softmax_topk(P, F32, 0, 64, 8, 0, P, BF16, P, None) == OK
    assert lib.om_route_softmax_topk(None, F32, 8, 64, 8, 0, P, BF16, P, None) == NULL
    assert lib.om_route_softmax_topk_bwd(P, F32, None, P, BF16, 8, 64, 8, 0, P, None) == NULL
    assert lib.om_route_sigmoid_group_topk(P, P, 8, 256, 7, 4, 8, 1, 2.5, P, P, None) == SHAPE   # 256 % 7
    assert lib.om_route_sigmoid_group_topk(P, None, 8, 256, 8, 4, 8, 1, 2.5, P, P, None) == NULL
    assert lib.om_router_gate_softmax_topk(P, P, 8, 2048, 300, 8, 0, P, P, BF16, P, None) == SHAPE   # N > 256
    assert lib.om_router_gate_softmax_topk(P, P, 8, 2000, 64, 8, 0, P, P, BF16, P, None) == SHAPE   # H % 512
    assert lib.om_router_gate_softmax_topk(ODD, P, 8, 2048, 64, 8, 0, P, P, BF16, P, None) == ALIGN
    assert lib.om_router_gate_softmax_topk(P, P, 8, 2048, 64, 8, 0, P, None, BF16, P, None) == NULL
    assert lib.om_router_gate_logits(P, P, 8, 2048, 64, None, None) == NULL
    need = lib.om_router_gate_logits_split_workspace_bytes(8192, 7168, 256)
    assert need > 0 and need % 16 == 0
    assert lib.om_router_gate_logits_split_workspace_bytes(8192, 7100, 256) == SHAPE     # H % 8
    assert lib.om_router_gate_logits_split_workspace_bytes(8192, 7168, 300) == SHAPE     # N > 256
    assert lib.om_router_gate_logits_split(P, P, 8192, 7168, 256, P, P, need - 1, None) == WORKSPACE
    assert lib.om_router_gate_logits_split(P, None, 8192, 7168, 256, P, P, need, None) == NULL
    assert lib.om_router_gate_logits_split(ODD, P, 8192, 7168, 256, P, P, need, None) == ALIGN
    assert lib.om_router_gate_logits_split(P, P, 0, 7168, 256, P, P, 0, None) == OK
    need = lib.om_router_gate_wgrad_workspace_bytes(16384, 2048, 64)
    assert need > 0 and need % 16 == 0
    assert lib.om_router_gate_wgrad_workspace_bytes(16384, 2044, 64) == SHAPE      # H % 8
    assert lib.om_router_gate_wgrad_workspace_bytes(16384, 2048, 300) == SHAPE     # more than 256 experts
    assert lib.om_router_gate_wgrad_workspace_bytes(16384, 2048, 48) > 0           # any expert count up to 256
    assert lib.om_router_gate_wgrad(P, P, 16384, 2048, 64, P, 7, P, need, None) == DTYPE
    assert lib.om_router_gate_wgrad(P, P, 16384, 2048, 0, P, BF16, P, need, None) == SHAPE
    assert lib.om_router_gate_dgrad(P, P, None, P, 16384, 2044, 64, None) == SHAPE      # H % 8
    assert lib.om_router_gate_dgrad(P, P, None, P, 16384, 2048, 257, None) == SHAPE
    assert lib.om_router_gate_dgrad(P, None, None, P, 16384, 2048, 64, None) == NULL
    assert lib.om_router_gate_dgrad(P, P, ODD, P, 16384, 2048, 64, None) == ALIGN
    assert lib.om_router_gate_dgrad(None, None, None, None, 0, 2048, 64, None) == OK
    assert lib.om_grad_scale(P, 100, 7, P, None) == DTYPE
    assert lib.om_grad_scale(P, 100, BF16, None, None) == NULL
    assert lib.om_grad_scale(ODD, 100, BF16, P, None) == ALIGN
    assert lib.om_grad_scale(None, 0, BF16, None, None) == OK
    assert lib.om_shard_clip_multiplier(P, 0, 7, 1.0, P, P, None) == DTYPE
    assert lib.om_shard_clip_multiplier(P, 2, BF16, 1.0, P, P, None) == SHAPE
    assert lib.om_shard_clip_multiplier(None, 0, BF16, 1.0, P, P, None) == NULL
    assert lib.om_shard_clip_multiplier(P, 1, BF16, 1.0, P, None, None) == NULL
    assert lib.om_adamw_traffic_probe(P, P, P, None, P, 1024, None) == NULL
    assert lib.om_router_balance_stats_masked(P, 7, P, 100, 64, 8, P, P, P, 1 << 20, None) == DTYPE
    assert lib.om_router_balance_stats_masked(P, F32, None, 100, 64, 65, P, P, P, 1 << 20, None) == SHAPE
    assert lib.om_router_balance_stats_masked(P, F32, P, 100, 64, 8, P, P, P, 8, None) == WORKSPACE
    assert lib.om_router_balance_bwd_masked(P, F32, None, P, 100, 64, P, None) == NULL
    assert lib.om_router_balance_bwd_masked(None, F32, None, None, 0, 64, None, None) == OK
    assert lib.om_router_gate_wgrad(P, P, 16384, 2048, 64, None, BF16, P, need, None) == NULL
    assert lib.om_router_gate_wgrad(P, None, 16384, 2048, 64, P, BF16, P, need, None) == NULL
    assert lib.om_router_gate_wgrad(P, P, 16384, 2048, 64, ODD, BF16, P, need, None) == ALIGN
    assert lib.om_router_gate_wgrad(P, P, 16384, 2048, 64, P, BF16, P, need - 1, None) == WORKSPACE


def test_sort_and_index_ops(lib):
    need = lib.om_moe_sort_workspace_bytes(1024, 8, 64)
    assert need > 0
    assert lib.om_moe_sort(P, 5, 1024, 8, 0, 64, P, P, P, P, P, P, need, None) == DTYPE
    assert lib.om_moe_sort(P, I64, 1024, 0, 0, 64, P, P, P, P, P, P, need, None) == SHAPE
    assert lib.om_moe_sort(P, I64, 1024, 8, 0, 64, None, P, P, P, P, P, need, None) == NULL
    assert lib.om_moe_sort(P, I64, 1024, 8, 0, 64, P, P, P, P, P, P, need - 1, None) == WORKSPACE
    assert lib.om_compute_partial_token_counts(P, I64, P, P, 0, 64, 1000, 8, 64, None) == SHAPE   # T % TH
    assert lib.om_index_gather(P, P, P, 16, 64, 3, None) == DTYPE
    assert lib.om_index_gather(P, None, P, 16, 64, BF16, None) == NULL
    assert lib.om_index_gather(P, P, P, 0, 64, BF16, None) == OK
    assert lib.om_index_add(P, P, P, -1, 64, BF16, None) == SHAPE
    assert lib.om_swiglu_fwd(P, P, ODD, 64, BF16, None) == ALIGN
    assert lib.om_swiglu_bwd(P, P, P, None, P, 64, BF16, None) == NULL


def test_rmsnorm_and_balance(lib):
    assert lib.om_rmsnorm_fwd(P, None, P, 1e-5, P, None, None, 8, 2048, 3, None) == DTYPE
    assert lib.om_rmsnorm_fwd(P, None, P, 1e-5, P, None, None, 8, 2052, BF16, None) == SHAPE   # E % 8
    assert lib.om_rmsnorm_fwd(P, None, P, 1e-5, P, None, None, 0, 2048, BF16, None) == OK
    assert lib.om_rmsnorm_fwd(P, None, None, 1e-5, P, None, None, 8, 2048, BF16, None) == NULL
    assert lib.om_rmsnorm_fwd(P, ODD, P, 1e-5, P, None, None, 8, 2048, BF16, None) == ALIGN
    need = lib.om_rmsnorm_bwd_workspace_bytes(300, 2048)
    assert need == 3 * 2048 * 4
    assert lib.om_rmsnorm_bwd(P, P, P, P, P, P, P, need - 1, 300, 2048, BF16, None) == WORKSPACE
    assert lib.om_rmsnorm_bwd(P, P, P, None, P, P, P, need, 300, 2048, BF16, None) == NULL
    need = lib.om_router_balance_workspace_bytes(1000, 64)
    assert lib.om_router_balance_stats(P, F32, 1000, 64, 8, P, P, P, need - 1, None) == WORKSPACE
    assert lib.om_router_balance_stats(P, 9, 1000, 64, 8, P, P, P, need, None) == DTYPE
    assert lib.om_router_balance_bwd(P, F32, None, 1000, 64, P, None) == NULL


def test_combine_with_residual(lib):
    args = (16384, 8, 2048, BF16, BF16, None)
    assert lib.om_reduce_ggemm_output_residual(P, P, P, P, P, None, P, *args) == NULL        # no residual
    assert lib.om_reduce_ggemm_output_residual(P, P, P, P, P, P, None, *args) == NULL
    assert lib.om_reduce_ggemm_output_residual(P, P, P, P, P, P, P, 16384, 8, 2048, 7, BF16, None) == DTYPE
    assert lib.om_reduce_ggemm_output_residual(P, P, P, P, P, None, P, 0, 8, 2048, BF16, BF16, None) == OK


def test_grouped_gemms(lib):
    args = (131072, 64, 2048, 1024, 0, None)
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 131072, 64, 2004, 1024, 0, None) == SHAPE    # N % 8
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 131072, 64, 2048, 1020, 0, None) == SHAPE    # K % 8
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 0, 64, 2048, 1024, 0, None) == OK            # no rows
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 4096, 1025, 256, 256, 0, None) == SHAPE      # G > 1024 (LDS table)
    assert lib.om_grouped_gemm_fwd(P, None, P, P, *args) == NULL
    assert lib.om_grouped_gemm_fwd(P, P, ODD, P, *args) == ALIGN
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 1 << 30, 64, 2048, 1024, 0, None) == SHAPE   # 2^40 elements or more
    assert lib.om_grouped_gemm_fwd(P, P, P, P, 4096, 64, 2048, 1024, 2048 * 1024 + 4, None) == ALIGN   # expert pitch % 8
    assert lib.om_grouped_gemm_dgrad(P, P, P, None, *args) == NULL
    assert lib.om_grouped_gemm_wgrad(P, P, P, P, 131072, 0, 2048, 1024, 0, None) == SHAPE   # G < 1
    assert lib.om_merged_mlp_gate_up_fwd(P, P, P, P, P, P, P, 131072, 64, 1004, 2048, 0, None) == SHAPE
    assert lib.om_merged_mlp_gate_up_fwd(P, P, None, P, P, P, P, 131072, 64, 1024, 2048, 0, None) == NULL
    assert lib.om_merged_mlp_down_dgrad(P, P, P, P, P, ODD, P, 131072, 64, 1024, 2048, 0, None) == ALIGN
    assert lib.om_merged_mlp_gate_up_dgrad(P, P, P, P, None, P, 131072, 64, 1024, 2048, 0, None) == NULL
    # float32 forms: N, K multiples of 8
    assert lib.om_grouped_gemm_fwd_f32(P, P, P, P, 4096, 8, 100, 256, 0, None) == SHAPE
    assert lib.om_grouped_gemm_fwd_f32(P, P, P, P, 0, 8, 64, 256, 0, None) == OK
    assert lib.om_grouped_gemm_fwd_f32(P, P, P, None, 4096, 8, 64, 256, 0, None) == NULL
    assert lib.om_grouped_gemm_fwd_f32(P, P, P, P, 4096, 8, 64, 256, 64 * 256 + 2, None) == ALIGN   # pitch % 4
    assert lib.om_grouped_gemm_dgrad_f32(P, ODD, P, P, 4096, 8, 64, 256, 0, None) == ALIGN
    assert lib.om_grouped_gemm_wgrad_f32(P, P, None, P, 4096, 8, 64, 256, 0, None) == NULL
    assert lib.om_grouped_gemm_wgrad_f32(P, P, P, P, 4096, 70000, 64, 256, 0, None) == SHAPE        # grid limit
    # the forms that read the tokens through an index
    g = (131072, 64, 1024, 2048, 0, None)
    assert lib.om_merged_mlp_gate_up_fwd_gathered(P, None, 16384, P, P, P, P, P, P, *g) == NULL      # no index
    assert lib.om_merged_mlp_gate_up_fwd_gathered(P, P, 0, P, P, P, P, P, P, *g) == SHAPE            # no source rows
    assert lib.om_merged_mlp_gate_up_fwd_gathered(P, P, 1 << 20, P, P, P, P, P, P, *g) == SHAPE      # indexed source of 2^31 elements or more
    assert lib.om_merged_mlp_gate_up_fwd_gathered(P, None, 0, P, P, P, P, P, P, 0, 64, 1024, 2048, 0, None) == OK
    assert lib.om_grouped_gemm_wgrad_gathered(P, P, None, 16384, P, P, *g) == NULL
    assert lib.om_grouped_gemm_wgrad_gathered(P, P, P, 0, P, P, *g) == SHAPE
    assert lib.om_grouped_gemm_wgrad_gathered(P, P, P, 16384, ODD, P, *g) == ALIGN


def test_router_that_sorts(lib):
    fits = lib.om_router_gate_softmax_topk_sort_fits
    assert fits(1, 2048, 64, 8) == 1 and fits(64, 2048, 64, 16) == 1
    for T, H, N, K in ((65, 2048, 64, 8), (0, 2048, 64, 8), (1, 2044, 64, 8), (1, 2048, 65, 8), (1, 2048, 64, 17), (1, 256, 8, 2), (1, 512, 64, 8)):
        assert fits(T, H, N, K) == 0
    f = lib.om_router_gate_softmax_topk_sort
    head, index = (P, P, 1, 2048, 64, 8, 0, P, BF16, P, BF16, P), (P,) * 6
    assert f(*head, 0, 65, *index, P, 1 << 20, None) == SHAPE
    assert f(*head, 8, 8, *index, P, 1 << 20, None) == SHAPE
    assert f(P, P, 65, *head[3:], 0, 64, *index, P, 1 << 20, None) == SHAPE
    assert f(*head[:8], 7, *head[9:], 0, 64, *index, P, 1 << 20, None) == DTYPE
    assert f(*head, 0, 64, P, P, None, P, P, P, P, 1 << 20, None) == NULL
    assert f(ODD, *head[1:], 0, 64, *index, P, 1 << 20, None) == ALIGN
    assert f(*head, 0, 64, *index, P, 16, None) == WORKSPACE


def test_router_backward_in_one_call(lib):
    need = lib.om_router_softmax_bwd_workspace_bytes(2048, 256, 8)
    assert need > 0
    for T, H, N in ((0, 256, 8), (64, 12, 8), (64, 256, 65)):
        assert lib.om_router_softmax_bwd_workspace_bytes(T, H, N) == SHAPE
    f = lib.om_router_softmax_bwd
    tail = (2048, 256, 8, 2, 1)
    assert f(P, P, P, F32, P, P, BF16, None, None, P, P, BF16, 2048, 256, 8, 9, 1, P, 1 << 30, None) == SHAPE
    assert f(P, P, P, 7, P, P, BF16, None, None, P, P, BF16, *tail, P, 1 << 30, None) == DTYPE
    assert f(P, P, P, F32, None, P, BF16, None, None, P, P, BF16, *tail, P, 1 << 30, None) == NULL
    assert f(P, P, P, F32, P, P, BF16, None, ODD, P, P, BF16, *tail, P, 1 << 30, None) == ALIGN
    assert f(P, P, P, F32, P, P, BF16, None, None, P, P, BF16, *tail, P, need - 1, None) == WORKSPACE


def test_routing_weight_folded_into_the_expert_mlp(lib):
    g = (131072, 64, 1024, 2048, 0, None)
    assert lib.om_moe_row_weights(P, P, P, P, P, 131072, 8, 7, None) == DTYPE
    assert lib.om_moe_row_weights(P, P, P, P, None, 131072, 8, F32, None) == NULL
    assert lib.om_moe_row_weights(P, P, P, P, P, 131072, 0, F32, None) == SHAPE
    assert lib.om_moe_row_weights(None, None, None, None, None, 0, 8, BF16, None) == OK
    assert lib.om_merged_mlp_gate_up_fwd_weighted(P, P, 16384, P, P, None, P, P, P, P, *g) == NULL   # no weights
    assert lib.om_merged_mlp_gate_up_fwd_weighted(P, None, 16384, P, P, P, P, P, P, P, *g) == NULL   # no index
    assert lib.om_merged_mlp_gate_up_fwd_weighted(P, P, 0, P, P, P, P, P, P, P, *g) == SHAPE
    assert lib.om_merged_mlp_gate_up_fwd_weighted(P, P, 16384, P, P, P, P, P, P, P, 131072, 64, 1004, 2048, 0, None) == SHAPE
    assert lib.om_merged_mlp_gate_up_fwd_weighted(P, None, 0, P, P, None, P, P, P, P, 0, 64, 1024, 2048, 0, None) == OK
    assert lib.om_sum_ggemm_output(P, None, P, None, P, 16384, 2048, BF16, None) == NULL
    assert lib.om_sum_ggemm_output(P, P, P, None, P, 16384, 2048, 7, None) == DTYPE
    assert lib.om_sum_ggemm_output(P, P, P, None, P, 0, 2048, BF16, None) == OK
    gw = (131072, 64, 2048, 1024, 0, None)
    assert lib.om_grouped_gemm_wgrad_gathered_out(P, None, 16384, P, P, P, *gw) == NULL
    assert lib.om_grouped_gemm_wgrad_gathered_out(P, P, 0, P, P, P, *gw) == SHAPE
    assert lib.om_grouped_gemm_wgrad_gathered_out(P, P, 1 << 21, P, P, P, *gw) == SHAPE   # indexed source of 2^31 elements or more
    assert lib.om_grouped_gemm_wgrad_gathered_out(P, P, 16384, P, ODD, P, *gw) == ALIGN
    assert lib.om_merged_mlp_row_dot_parts(1024) == 16
    assert lib.om_merged_mlp_row_dot_parts(200) == 4      # partial last 64-column group
    assert lib.om_merged_mlp_row_dot_parts(100) == SHAPE
    assert lib.om_merged_mlp_down_dgrad_weighted(P, P, 16384, P, P, P, P, P, P, None, P, *g) == NULL   # no row_dot
    assert lib.om_merged_mlp_down_dgrad_weighted(P, P, 16384, P, P, P, None, P, P, P, P, *g) == NULL   # no weights
    assert lib.om_merged_mlp_down_dgrad_weighted(P, None, 16384, P, P, P, P, P, P, P, P, *g) == NULL   # no index
    assert lib.om_merged_mlp_down_dgrad_weighted(P, P, 0, P, P, P, P, P, P, P, P, *g) == SHAPE
    assert lib.om_merged_mlp_down_dgrad_weighted(P, P, 16384, P, P, P, P, ODD, P, P, P, *g) == ALIGN
    assert lib.om_merged_mlp_down_dgrad_weighted(P, None, 0, P, P, P, None, P, P, None, P, 0, 64, 1024, 2048, 0, None) == OK
    assert lib.om_moe_row_weights_grad(P, 0, P, P, P, P, 131072, 8, F32, None) == SHAPE
    assert lib.om_moe_row_weights_grad(None, 16, P, P, P, P, 131072, 8, F32, None) == NULL
    assert lib.om_moe_row_weights_grad(P, 16, P, P, P, P, 131072, 8, 9, None) == DTYPE
    assert lib.om_moe_row_weights_grad(None, 16, None, None, None, None, 0, 8, F32, None) == OK
    sums = lib.om_sum_ggemm_output_row_weights_grad
    assert sums(P, None, P, None, P, 16384, 2048, BF16, P, 16, 131072, P, P, 8, BF16, None) == NULL
    assert sums(P, P, P, None, P, 16384, 2048, BF16, None, 16, 131072, P, P, 8, BF16, None) == NULL
    assert sums(P, P, P, None, P, 16384, 2048, BF16, P, 16, 131072, P, None, 8, BF16, None) == NULL
    assert sums(P, P, P, None, P, 16384, 2048, BF16, P, 0, 131072, P, P, 8, BF16, None) == SHAPE
    assert sums(P, P, P, None, P, 16384, 2048, BF16, P, 16, 131072, P, P, 0, BF16, None) == SHAPE
    assert sums(P, P, P, None, P, 16384, 2048, 7, P, 16, 131072, P, P, 8, BF16, None) == DTYPE
    assert sums(P, P, P, None, P, 16384, 2048, BF16, P, 16, 131072, P, P, 8, 7, None) == DTYPE
    assert sums(None, None, None, None, None, 0, 2048, BF16, None, 16, 0, None, None, 8, BF16, None) == OK


def test_products_over_a_bound_of_the_rows(lib):
    """0 <= expected_rows <= rows; everything else as the plain forms."""
    for expected in (-1, 4097):
        assert lib.om_grouped_gemm_fwd_bound(P, P, P, P, 4096, expected, 64, 2048, 1024, 0, None) == SHAPE
        assert lib.om_merged_mlp_gate_up_fwd_weighted_bound(P, P, 512, P, P, P, P, P, P, P, 4096, expected, 64, 1024, 2048, 0,
                                                            None) == SHAPE
        assert lib.om_merged_mlp_down_dgrad_weighted_bound(P, P, 512, P, P, P, P, P, P, P, P, 4096, expected, 64, 1024, 2048, 0,
                                                           None) == SHAPE
        assert lib.om_merged_mlp_gate_up_dgrad_bound(P, P, P, P, P, P, 4096, expected, 64, 1024, 2048, 0, None) == SHAPE
        for form in (lib.om_grouped_gemm_wgrad_merged_bound, lib.om_grouped_gemm_wgrad_merged_accumulate_bound):
            assert form(P, P, P, P, P, P, P, 512, P, P, P, P, 4096, expected, 64, 1024, 2048, 0, 0, 0, None) == SHAPE
    assert lib.om_grouped_gemm_fwd_bound(P, None, P, P, 4096, 64, 64, 2048, 1024, 0, None) == NULL
    assert lib.om_grouped_gemm_fwd_bound(None, None, None, None, 0, 0, 64, 2048, 1024, 0, None) == OK
    assert lib.om_merged_mlp_gate_up_fwd_weighted_bound(P, None, 512, P, P, P, P, P, P, P, 4096, 64, 64, 1024, 2048, 0,
                                                        None) == NULL
    assert lib.om_merged_mlp_down_dgrad_weighted_bound(P, P, 512, P, P, P, P, P, ODD, P, P, 4096, 64, 64, 1024, 2048, 0,
                                                       None) == ALIGN
    assert lib.om_grouped_gemm_wgrad_merged_bound(P, P, P, P, P, P, P, 512, P, P, None, P, 4096, 64, 64, 1024, 2048, 0, 0, 0, None) == NULL
    assert lib.om_grouped_gemm_wgrad_merged_accumulate_bound(P, P, P, P, P, P, P, 512, P, ODD, P, P, 4096, 64, 64, 1024, 2048, 0, 0, 0,
                                                             None) == ALIGN
    assert lib.om_merged_mlp_gate_up_dgrad_bound(P, P, P, P, None, P, 4096, 64, 64, 1024, 2048, 0, None) == NULL


def _dense(rows=64, a=(P, P), w=(P, P), c=(P, P, P), g=P, u=P, cum=P):
    """An om_dense_expert."""
    return ctypes.create_string_buffer(struct.pack("10Qq", *(v or 0 for v in (*a, *w, *c, g, u, cum)), rows))


# entry point, arguments ahead of cum_token_counts, extents, fields of the dense expert that it reads (a, w, c, whether g and u)
DENSE = [("om_merged_mlp_gate_up_fwd_weighted_dense", (P, P, 64, P, P, P, P, P, P), (1, 2, 3, False)),
         ("om_grouped_gemm_fwd_dense", (P, P, P), (1, 1, 1, False)),
         ("om_merged_mlp_down_dgrad_weighted_dense", (P, P, 64, P, P, P, P, P, P, P), (1, 1, 2, True)),
         ("om_merged_mlp_gate_up_dgrad_dense", (P, P, P, P, P), (2, 2, 1, False))]


@pytest.mark.parametrize("name,args,fields", DENSE)
def test_products_with_a_dense_expert(lib, name, args, fields):
    """What the routed operands are refused for in the plain forms, and the dense expert's own; it rides at these sizes."""
    n_a, n_w, n_c, gu = fields

    def call(dense, args=args, rows=512, expected=128, G=32, I=1024, H=2048, stride=0):
        return getattr(lib, name)(*args, P, rows, expected, G, I, H, stride, ctypes.addressof(dense) if dense is not None else None, None)

    assert lib.om_merged_mlp_dense_products(128, 32, 1024, 2048, 64) == 15
    assert call(None) == NULL
    assert call(_dense(), expected=513) == SHAPE and call(_dense(), expected=-1) == SHAPE
    assert call(_dense(), I=1004) == SHAPE and call(_dense(), H=2044) == SHAPE and call(_dense(), G=0) == SHAPE
    assert call(_dense(), stride=1024 * 2048 + 4) == ALIGN
    assert call(_dense(rows=0)) == SHAPE and call(_dense(rows=1 << 31)) == SHAPE
    assert call(_dense(cum=None)) == NULL
    for field, count in (("a", n_a), ("w", n_w), ("c", n_c)):
        size = {"a": 2, "w": 2, "c": 3}[field]
        for i in range(count):
            assert call(_dense(**{field: [None if j == i else P for j in range(size)]})) == NULL, (field, i)
            assert call(_dense(**{field: [ODD if j == i else P for j in range(size)]})) == ALIGN, (field, i)
    if gu:
        assert call(_dense(g=None)) == NULL and call(_dense(u=ODD)) == ALIGN
    for i, v in enumerate(args):
        if v == P:
            assert call(_dense(), args[:i] + (None,) + args[i + 1:]) == NULL, i
    if name != "om_merged_mlp_down_dgrad_weighted_dense":   # (its last is of 32 bits)
        assert call(_dense(), args[:-1] + (ODD,)) == ALIGN


def test_dense_products(lib):
    for bad in ((-1, 8, 1024, 1024, 64), (64, 0, 1024, 1024, 64), (64, 8, 1004, 1024, 64), (64, 8, 1024, 1004, 64), (64, 8, 1024, 1024, 0)):
        assert lib.om_merged_mlp_dense_products(*bad) == SHAPE and lib.om_merged_mlp_dense_rides(*bad) == SHAPE
    for sizes in ((64, 32, 2048, 7168, 64), (8192, 32, 2048, 7168, 8192), (5000, 32, 1000, 1200, 5000)):
        assert lib.om_merged_mlp_dense_rides(*sizes) == lib.om_merged_mlp_dense_products(*sizes) & 1


def test_check_raises_with_the_library_text():
    with pytest.raises(n.NativeLibraryError, match="dtype"):
        n.check(DTYPE, "om_adamw_step")
