"""GPU parity of the dense bf16 GEMM (gemm_graphsafe_cuda / gemm_cuda, the
Kimi shared expert's projections; linear.cu:321-344) and of the whole Kimi
decode layer with its shared expert and residual join (moe_nccl.rs:98-239),
against the CPU oracle.  Tolerance: |gpu - ref| <= 1e-3 + 1e-2 |ref| (the
library sums K in its own order); exact where every partial sum is exact."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_helpers import assert_bf16_close, dev, host

pytestmark = pytest.mark.gpu


def _gemm(w, x):
    from pegainfer_amd import ops
    y = torch.zeros(x.shape[0], w.shape[0], dtype=torch.bfloat16, device="cuda")
    ops.gemm_graphsafe(dev(w), dev(x), y)
    return host(y)


@pytest.mark.parametrize("M,N,K", [(4096, 64, 7168), (7168, 64, 2048), (64, 1, 32),
                                   (48, 7, 96), (256, 33, 512), (128, 100, 256), (16, 200, 64),
                                   (2048, 17, 1024)])
def test_dense_gemm_matches_oracle(oracle, M, N, K):
    g = np.random.default_rng(M * 131 + N * 7 + K)
    w = oracle.f32_to_bf16((g.standard_normal((M, K)) * 0.02).astype(np.float32))
    x = oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32))
    assert_bf16_close(_gemm(w, x), oracle.dense_gemm(w, x), what=f"dense {M}x{N}x{K}")


def test_dense_gemm_exact_when_partial_sums_are_exact(oracle):
    g = np.random.default_rng(3)
    M, N, K = 96, 40, 640
    w = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 2, (M, K)))
                           .astype(np.float32))
    x = oracle.f32_to_bf16(g.integers(-6, 7, (N, K)).astype(np.float32))
    assert np.array_equal(_gemm(w, x), oracle.dense_gemm(w, x))


def test_dense_gemm_one_hot_rows_give_weight_columns(oracle):
    g = np.random.default_rng(4)
    M, K = 160, 256
    w = oracle.f32_to_bf16(g.standard_normal((M, K)).astype(np.float32))
    ks = [0, 31, 32, 200, 255]
    x = np.zeros((len(ks), K), np.uint16)
    for n, k in enumerate(ks):
        x[n, k] = 0x3F80  # bf16 1.0
    y = _gemm(w, x)
    for n, k in enumerate(ks):
        assert np.array_equal(y[n], w[:, k])


def test_dense_gemm_entry_points_agree_and_reject(oracle):
    from pegainfer_amd import _lib
    g = np.random.default_rng(5)
    M, N, K = 64, 9, 128
    w = dev(oracle.f32_to_bf16(g.standard_normal((M, K)).astype(np.float32)))
    x = dev(oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32)))
    y1 = torch.zeros(N, M, dtype=torch.bfloat16, device="cuda")
    y2 = torch.zeros_like(y1)
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert L.gemm_cuda(p(w), p(x), p(y1), M, N, K, s) == 0
    assert L.gemm_graphsafe_cuda(p(w), p(x), p(y2), M, N, K, s) == 0
    assert np.array_equal(host(y1), host(y2))
    assert L.gemm_graphsafe_cuda(p(w), p(x), p(y2), 40, N, K, s) == 801    # M % 16
    assert L.gemm_graphsafe_cuda(p(w), p(x), p(y2), M, N, 100, s) == 801   # K % 32
    assert L.gemm_graphsafe_cuda(None, p(x), p(y2), M, N, K, s) == 1
    assert L.gemm_graphsafe_cuda(p(w), p(x), p(y2), M, 0, K, s) == 1


@pytest.mark.parametrize("T", [24, 3, 600])
def test_kimi_decode_layer_with_shared_expert(oracle, T):
    """Shared expert (bf16 gate/up and down), router select, routed experts and
    the residual join, against the oracle's chain of the same stages.  At 3 tokens
    the layer routes through the fused select + permutation launch in one workgroup,
    at 24 in several, and at 600 (4800 routes) through the two launches."""
    from pegainfer_amd import layer, ops, synth
    E, H, I, SI = 48, 1024, 256, 512
    assert layer.fused_route(T, 8, 384) == (T != 600)
    g = synth.rng(11, T)
    gate, up, down = (synth.int4_checkpoint(g, E, I, H), synth.int4_checkpoint(g, E, I, H),
                      synth.int4_checkpoint(g, E, H, I))
    gu = oracle.f32_to_bf16((g.standard_normal((2 * SI, H)) * 0.03).astype(np.float32))
    dn = oracle.f32_to_bf16((g.standard_normal((H, SI)) * 0.03).astype(np.float32))
    hidden = synth.normal_bf16(g, (T, H))
    normed = synth.normal_bf16(g, (T, H))
    logits = g.standard_normal((T, 384), dtype=np.float32)
    bias = np.zeros(384, np.float32)
    routed = layer.RoutedExperts(layer.package_w13(gate, up), layer.package_projection(*down),
                                 max_tokens=T, topk=8, block_size=ops.kimi_marlin_block_size(T))
    shared = layer.KimiSharedExpert(dev(gu), dev(dn), max_tokens=T)
    moe = layer.KimiMoeDecodeLayer(routed, shared)
    out = torch.zeros(T, H, dtype=torch.bfloat16, device="cuda")
    moe.forward(dev(hidden), dev(normed), dev(logits), dev(bias), out)
    # the oracle's chain
    idx, w = oracle.kimi_router(logits, bias, 8, 1.0)
    assert np.array_equal(host(moe.topk_idx), idx)
    proj = oracle.dense_gemm(dn, oracle.swiglu(oracle.dense_gemm(gu, normed), SI))
    assert_bf16_close(host(moe.projected), proj, what="shared expert projected")
    w13p = np.concatenate([gate[0], up[0]], axis=1)
    w13s = np.concatenate([gate[1], up[1]], axis=1)
    routed_ref, _ = oracle.kimi_moe_layer(normed, w13p, w13s, down[0], down[1], idx.reshape(-1),
                                          w, global_start=0, local_experts=E,
                                          block_size=routed.block_size, hidden=H, inter=I)
    # the routed branch against the oracle's fp32 layer output, at the routed-layer bound
    rg, rr = host(moe.routed_f32).astype(np.float64), routed_ref.astype(np.float64)
    assert (np.abs(rg - rr) <= 2e-3 + 2e-2 * np.abs(rr)).all(), "routed branch"
    if T <= 24:
        # two GEMM chains of the same tolerance composed: twice the per-GEMM bound (over
        # 600 x 1024 outputs the routed error, scaled by 2.827 in the join, reaches that
        # bound's tail near zero, so the larger case checks the stages instead)
        ref = oracle.residual_add_scaled_f32(hidden, proj, routed_ref, ops.KIMI_K2_ROUTER_SCALE)
        assert_bf16_close(host(out), ref, rtol=2e-2, atol=2e-3, what="Kimi decode layer")
    # the join itself is exact given its inputs
    assert np.array_equal(host(out), oracle.residual_add_scaled_f32(
        hidden, host(moe.projected), host(moe.routed_f32), ops.KIMI_K2_ROUTER_SCALE))


@pytest.mark.parametrize("I,N,K", [(2048, 64, 7168), (256, 24, 1024), (48, 7, 96), (16, 100, 64)])
def test_dense_w13_swiglu_equals_gemm_then_swiglu(oracle, I, N, K):
    """The fused launch against the two-call chain it replaces (gate/up GEMM to
    bf16, then the reference SwiGLU): the same bits.  The chain's GEMM is checked
    against the oracle above and its SwiGLU bit-exactly elsewhere."""
    from pegainfer_amd import ops
    g = np.random.default_rng(I * 31 + N * 5 + K)
    w = dev(oracle.f32_to_bf16((g.standard_normal((2 * I, K)) * 0.02).astype(np.float32)))
    x = dev(oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32)))
    w, x = w.view(torch.bfloat16), x.view(torch.bfloat16)
    gu = torch.zeros(N, 2 * I, dtype=torch.bfloat16, device="cuda")
    ops.gemm_graphsafe(w, x, gu)
    chain = torch.zeros(N, I, dtype=torch.bfloat16, device="cuda")
    ops.kimi_marlin_w13_swiglu(gu, chain, N, I)
    fused = torch.full((N, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.dense_w13_swiglu(w, x, fused)
    torch.cuda.synchronize()
    assert np.array_equal(host(fused), host(chain)), (I, N, K)


def test_dense_w13_swiglu_rejects():
    from pegainfer_amd import _lib
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    buf = torch.zeros(4096, dtype=torch.bfloat16, device="cuda")
    p = ctypes.c_void_p(buf.data_ptr())
    assert L.pega_dense_w13_swiglu(p, p, p, 24, 4, 64, s) == 801   # inter % 16
    assert L.pega_dense_w13_swiglu(p, p, p, 16, 4, 48, s) == 801   # K % 32
    assert L.pega_dense_w13_swiglu(None, p, p, 16, 4, 64, s) == 1
    torch.cuda.synchronize()


def _token_blocks(M, N, swiglu, cu):
    """The launcher's (workgroup rows, token blocks) choice, restated so that the
    shapes below provably reach the 3- and 4-token-block kernels (dense.hip)."""
    mr = 2 if swiglu else (2 if M % 32 == 0 else 1)
    gx = M // 16 if swiglu else M // (16 * mr)
    rb = 1 if N <= 16 else 2 if N <= 32 else 3 if N <= 48 else 4
    if rb > 1 and gx * -(-N // (16 * rb)) < cu:
        rb = (rb + 1) // 2
    return rb


@pytest.mark.parametrize("M,N,K,rb", [(7168, 256, 2048, 4), (8192, 40, 1024, 3),
                                      (4096, 100, 7168, 4), (8192, 48, 512, 3)])
def test_dense_gemm_three_and_four_token_blocks(oracle, M, N, K, rb):
    """Prefill-sized shared-expert shapes whose launches use 3 or 4 token blocks per
    workgroup (the D = 3 load ring and the larger reduction buffer)."""
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    assert _token_blocks(M, N, False, cu) == rb
    g = np.random.default_rng(M + N + K)
    w = oracle.f32_to_bf16((g.standard_normal((M, K)) * 0.02).astype(np.float32))
    x = oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32))
    assert_bf16_close(_gemm(w, x), oracle.dense_gemm(w, x), what=f"dense {M}x{N}x{K} rb={rb}")
    # exact operands: bit for bit
    we = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 0, (M, K)))
                            .astype(np.float32))
    xe = oracle.f32_to_bf16(g.integers(-3, 4, (N, K)).astype(np.float32))
    ref = oracle.bf16_to_f32(xe).astype(np.float32) @ oracle.bf16_to_f32(we).astype(np.float32).T
    assert np.array_equal(_gemm(we, xe), oracle.f32_to_bf16(ref))


@pytest.mark.parametrize("I,N,K,rb", [(2048, 256, 7168, 4), (4096, 40, 1024, 3)])
def test_dense_w13_swiglu_three_and_four_token_blocks(oracle, I, N, K, rb):
    from pegainfer_amd import ops
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    assert _token_blocks(I, N, True, cu) == rb
    g = np.random.default_rng(I + N + K)
    w = dev(oracle.f32_to_bf16((g.standard_normal((2 * I, K)) * 0.02).astype(np.float32)))
    x = dev(oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32)))
    fused = torch.full((N, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.dense_w13_swiglu(w, x, fused)
    if N < 256:
        # the two-call chain runs the same GEMM kernel: the same bits
        gu = torch.zeros(N, 2 * I, dtype=torch.bfloat16, device="cuda")
        ops.gemm_graphsafe(w, x, gu)
        chain = torch.zeros(N, I, dtype=torch.bfloat16, device="cuda")
        ops.kimi_marlin_w13_swiglu(gu, chain, N, I)
        assert np.array_equal(host(fused), host(chain))
    else:
        # from 256 tokens gemm_graphsafe takes hipBLASLt (another summation order): the
        # fused launch against the oracle's GEMM + SwiGLU on sampled tokens instead
        g2 = np.random.default_rng(1)
        rows = np.unique(np.concatenate([[0, N - 1], g2.integers(0, N, 14)]))
        ref = oracle.swiglu(oracle.dense_gemm(host(w), host(x)[rows]), I)
        assert_bf16_close(host(fused)[rows], ref, what="fused dense SwiGLU")


@pytest.mark.parametrize("M,N,K", [(7168, 64, 2048), (4096, 57, 1024)])
def test_dense_gemm_decode_sized_token_halves(oracle, M, N, K):
    """Decode-sized token counts split into two 32-token workgroups with the short-K,
    few-waves launch (dense.hip): the Kimi shared expert's down GEMM at 64 tokens, and
    57 tokens (a partial last token block).  Random operands within the tolerance,
    exact operands bit for bit."""
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    assert _token_blocks(M, N, False, cu) == 2
    g = np.random.default_rng(M + N + K)
    w = oracle.f32_to_bf16((g.standard_normal((M, K)) * 0.02).astype(np.float32))
    x = oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32))
    assert_bf16_close(_gemm(w, x), oracle.dense_gemm(w, x), what=f"dense {M}x{N}x{K}")
    we = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 0, (M, K)))
                            .astype(np.float32))
    xe = oracle.f32_to_bf16(g.integers(-3, 4, (N, K)).astype(np.float32))
    ref = oracle.bf16_to_f32(xe).astype(np.float32) @ oracle.bf16_to_f32(we).astype(np.float32).T
    assert np.array_equal(_gemm(we, xe), oracle.f32_to_bf16(ref))


@pytest.mark.parametrize("M,N,K", [(4096, 256, 1024), (2048, 300, 512), (7168, 512, 2048),
                                   (4096, 4096, 7168)])
def test_dense_gemm_prefill_sizes_sampled_rows(oracle, M, N, K):
    """From 256 tokens the dense GEMM runs on hipBLASLt; its rows against the oracle on a
    sample of tokens (the first, the last and a seeded spread), at the Kimi shared
    expert's gate/up shape at 4096 tokens among them."""
    g = np.random.default_rng(M + N + K)
    w = oracle.f32_to_bf16((g.standard_normal((M, K)) * 0.02).astype(np.float32))
    x = oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32))
    y = _gemm(w, x)
    rows = np.unique(np.concatenate([[0, N - 1], g.integers(0, N, 14)]))
    assert_bf16_close(y[rows], oracle.dense_gemm(w, x[rows]), what=f"dense {M}x{N}x{K}")


def test_dense_gemm_prefill_exact_when_partial_sums_are_exact(oracle):
    g = np.random.default_rng(13)
    M, N, K = 256, 320, 640
    w = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 2, (M, K)))
                           .astype(np.float32))
    x = oracle.f32_to_bf16(g.integers(-6, 7, (N, K)).astype(np.float32))
    assert np.array_equal(_gemm(w, x), oracle.dense_gemm(w, x))


def test_kimi_shared_expert_prefill_path(oracle):
    """The shared expert at 4096 tokens (gate/up GEMM, SwiGLU kernel, down GEMM: the
    reference's prefill sequence) against the oracle's chain on sampled tokens, and its
    replay in a HIP graph equal to the eager result."""
    from pegainfer_amd import layer
    g = np.random.default_rng(21)
    T, H, SI = 4096, 7168, 2048
    gu = oracle.f32_to_bf16((g.standard_normal((2 * SI, H)) * 0.02).astype(np.float32))
    dn = oracle.f32_to_bf16((g.standard_normal((H, SI)) * 0.02).astype(np.float32))
    normed = oracle.f32_to_bf16(g.standard_normal((T, H)).astype(np.float32))
    shared = layer.KimiSharedExpert(dev(gu), dev(dn), max_tokens=T)
    x = dev(normed)
    out = torch.zeros(T, H, dtype=torch.bfloat16, device="cuda")
    shared.forward(x, out)
    torch.cuda.synchronize()
    got = host(out)
    rows = np.unique(np.concatenate([[0, T - 1], g.integers(0, T, 6)]))
    # each stage against the oracle given the GPU's own input to it: the gate/up GEMM, the
    # SwiGLU (exact), the down GEMM
    h13 = host(shared.h13)[rows]
    assert_bf16_close(h13, oracle.dense_gemm(gu, normed[rows]), what="shared gate/up")
    act = host(shared.act)[rows]
    assert np.array_equal(act, oracle.swiglu(h13, SI))
    assert_bf16_close(got[rows], oracle.dense_gemm(dn, act), what="shared down")
    graph = layer.capture_graph(lambda: shared.forward(x, out))
    for _ in range(2):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(out), got)


@pytest.mark.parametrize("M,N,K", [(16, 33, 32), (48, 64, 96), (80, 65, 160), (112, 97, 224),
                                   (208, 129, 2080), (4096, 65, 512), (4096, 100, 96),
                                   (4096, 200, 352), (4096, 255, 64), (7168, 100, 160),
                                   (7168, 5, 160), (8192, 255, 288)])
def test_dense_tile_shapes_exact(oracle, M, N, K):
    """The LDS-tiled kernel's tile shapes (the shapes pick each of them) at ragged features,
    tokens and k chunks, with Y aligned to its stores and two bytes off; exact operands, so
    every summation order gives the fp32 product's bits."""
    from pegainfer_amd import _lib
    g = np.random.default_rng(M + N + K)
    w = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 0, (M, K)))
                           .astype(np.float32))
    x = oracle.f32_to_bf16(g.integers(-3, 4, (N, K)).astype(np.float32))
    ref = oracle.f32_to_bf16(oracle.bf16_to_f32(x) @ oracle.bf16_to_f32(w).T)
    wd, xd = dev(w), dev(x)
    for off in (0, 1):
        y = torch.full((N * M + 2,), 7.0, dtype=torch.bfloat16, device="cuda")
        _lib.call("gemm_graphsafe_cuda", wd.data_ptr(), xd.data_ptr(), y.data_ptr() + 2 * off, M, N,
                  K, torch.cuda.current_stream().cuda_stream)
        got = host(y)
        assert np.array_equal(got[off:off + N * M].reshape(N, M), ref), off
        assert (got[:off] == 0x40E0).all() and (got[off + N * M:] == 0x40E0).all()


@pytest.mark.parametrize("I,N,K", [(16, 33, 32), (48, 100, 160), (80, 129, 96), (2048, 70, 352),
                                   (2048, 255, 96), (2064, 160, 64)])
def test_dense_tile_swiglu_equals_gemm_then_swiglu(oracle, I, N, K):
    """Gate and up features of one tile, ragged in both halves: the bits of the two calls."""
    from pegainfer_amd import ops
    g = np.random.default_rng(I + N + K)
    w = dev(oracle.f32_to_bf16((g.standard_normal((2 * I, K)) * 0.1).astype(np.float32)))
    x = dev(oracle.f32_to_bf16(g.standard_normal((N, K)).astype(np.float32)))
    fused = torch.full((N, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.dense_w13_swiglu(w, x, fused)
    gu = torch.zeros(N, 2 * I, dtype=torch.bfloat16, device="cuda")
    ops.gemm_graphsafe(w, x, gu)
    chain = torch.zeros(N, I, dtype=torch.bfloat16, device="cuda")
    ops.kimi_marlin_w13_swiglu(gu, chain, N, I)
    assert np.array_equal(host(fused), host(chain))


@pytest.mark.parametrize("M,N,K", [(4096, 33, 32), (4096, 64, 288), (4096, 50, 800),
                                   (4128, 64, 1056), (4096, 64, 2080), (8192, 17, 576)])
def test_dense_tile_long_chunks_exact(oracle, M, N, K):
    """The 32 x 32 tile's chunks of 256 k: fewer chunks than its ring has stages, the ring come
    round, and a tail of every kind (a step, most of a chunk) at the ends of K's shares."""
    test_dense_tile_shapes_exact(oracle, M, N, K)
    test_dense_tile_swiglu_equals_gemm_then_swiglu(oracle, M // 2, N, K)


@pytest.mark.parametrize("N,K", [(33, 96), (100, 2080), (700, 160), (1500, 64), (4100, 32)])
def test_dense_tile_router_logits_exact(oracle, N, K):
    """The fp32 epilogue through the router entry point, on exact operands."""
    from pegainfer_amd import ops
    g = np.random.default_rng(N + K)
    M = 384
    w = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 0, (M, K)))
                           .astype(np.float32))
    x = oracle.f32_to_bf16(g.integers(-3, 4, (N, K)).astype(np.float32))
    logits = torch.zeros(N, M, device="cuda")
    tw = torch.zeros(N, 8, device="cuda")
    ti = torch.zeros(N, 8, dtype=torch.int32, device="cuda")
    ops.kimi_k2_router_noaux_tc(dev(x), dev(w), torch.zeros(M, device="cuda"), logits, tw, ti, N, N)
    assert np.array_equal(host(logits), oracle.bf16_to_f32(x) @ oracle.bf16_to_f32(w).T)


@pytest.mark.parametrize("M,N,K", [(16, 1, 32), (16, 17, 96), (48, 16, 128), (48, 33, 160),
                                   (384, 170, 2080), (2048, 32, 352), (2048, 33, 128),
                                   (4096, 31, 160), (5120, 16, 160), (7168, 9, 2368)])
def test_dense_stream_shapes_exact(oracle, M, N, K):
    """The streaming kernel at its least K (one wave; four waves of a step), at token blocks of
    16 and 32 with remainders, and on both sides of the line to the LDS-tiled kernel: plain
    and SwiGLU, on exact operands (every summation order gives the fp32 product's bits)."""
    from pegainfer_amd import ops
    g = np.random.default_rng(M + N + K)
    w = oracle.f32_to_bf16(np.ldexp(g.integers(-8, 8, (M, K)), g.integers(-4, 0, (M, K)))
                           .astype(np.float32))
    x = oracle.f32_to_bf16(g.integers(-3, 4, (N, K)).astype(np.float32))
    wd, xd = dev(w), dev(x)
    y = torch.full((N + 1, M), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.gemm_graphsafe(wd, xd, y[:N])
    ref = oracle.f32_to_bf16(oracle.bf16_to_f32(x) @ oracle.bf16_to_f32(w).T)
    assert np.array_equal(host(y[:N]), ref) and bool((y[N] == 7.0).all())
    if M % 32 == 0:
        fused = torch.full((N + 1, M // 2), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.dense_w13_swiglu(wd, xd, fused[:N])
        chain = torch.zeros(N, M // 2, dtype=torch.bfloat16, device="cuda")
        ops.kimi_marlin_w13_swiglu(y[:N], chain, N, M // 2)
        assert np.array_equal(host(fused[:N]), host(chain)) and bool((fused[N] == 7.0).all())


@pytest.mark.parametrize("M,N,K,shares", [
    (384, 1, 7168, 16), (384, 33, 7168, 16), (384, 400, 7168, 16),  # router logits
    (384, 1000, 7168, 2), (384, 4100, 4096, 2),
    (2048, 96, 2816, 16), (4096, 5, 7168, 16), (4096, 24, 7168, 2), (4096, 64, 7168, 2),
    (4096, 100, 4128, 2), (4096, 250, 7168, 2), (16384, 3, 16384, 8), (16384, 12, 4096, 2),
    (16384, 100, 8192, 4), (48, 17, 544, 16), (48, 200, 352, 8), (5120, 7, 5120, 16),
    (5120, 12, 5120, 16), (16384, 7, 4096, 2), (1024, 250, 4096, 2), (1024, 250, 8192, 4),
    (2048, 65, 2048, 16)])
def test_dense_sums_are_shares_of_k_in_order(oracle, M, N, K, shares):
    """The order of the fp32 sums: `shares` contiguous parts of K's 32-k steps, added in order.
    One nonzero k in each share makes a share's sum one exact product, and a large term that
    a later share cancels makes the order of the additions show in every output format, so the
    result equals the ordered fp32 sum bit for bit and another grouping's does not."""
    from pegainfer_amd import ops
    g = np.random.default_rng(M + N + K)
    steps = K // 32
    def bf16(*shape):
        return oracle.bf16_to_f32(oracle.f32_to_bf16(g.uniform(0.5, 1, shape).astype(np.float32)))
    if shares == 2:
        # share 0: big + a small term, which its chain's sum loses; share 1: -big, then a small
        # negative term, lost likewise
        half = steps // 2 * 32
        at = [0, 40, half + 16, half + 32 + (112 - half - 32) % 128]
        col, xs = bf16(M, 4), bf16(N, 4)
        col[:, 2] = col[:, 0]
        xs[:, 0], xs[:, 2] = 2.0 ** 30, -2.0 ** 30
        xs[:, 3] *= -1
        ref = np.zeros((N, M), np.float32)
    else:
        at = [32 * int(g.integers(steps * s // shares, steps * (s + 1) // shares))
              + int(g.integers(0, 32)) for s in range(shares)]
        col, xs = bf16(M, shares), bf16(N, shares)
        first, last = (int(v) for v in sorted(g.choice(shares, 2, replace=False)))
        col[:, last] = col[:, first]
        xs[:, first], xs[:, last] = 2.0 ** 20, -2.0 ** 20
        ref = np.zeros((N, M), np.float32)
        for s in range(shares):
            ref = ref + xs[:, s:s + 1] * col[:, s]
    w = torch.zeros(M, K, dtype=torch.bfloat16, device="cuda")
    x = torch.zeros(N, K, dtype=torch.bfloat16, device="cuda")
    w[:, at] = dev(col).to(torch.bfloat16)
    x[:, at] = dev(xs).to(torch.bfloat16)
    if M == 384:
        got = torch.zeros(N, M, device="cuda")
        ops.kimi_k2_router_noaux_tc(x, w, torch.zeros(M, device="cuda"), got,
                                    torch.zeros(N, 8, device="cuda"),
                                    torch.zeros(N, 8, dtype=torch.int32, device="cuda"), N, N)
        assert np.array_equal(host(got), ref)
    if N < 256:
        y = torch.zeros(N, M, dtype=torch.bfloat16, device="cuda")
        ops.gemm_graphsafe(w, x, y)
        assert np.array_equal(host(y), oracle.f32_to_bf16(ref))
        if M % 32 == 0:
            act = torch.zeros(N, M // 2, dtype=torch.bfloat16, device="cuda")
            ops.dense_w13_swiglu(w, x, act)
            chain = torch.zeros_like(act)
            ops.kimi_marlin_w13_swiglu(y, chain, N, M // 2)
            assert np.array_equal(host(act), host(chain))
