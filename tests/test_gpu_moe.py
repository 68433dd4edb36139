"""GPU parity: grouped GEMMs, fused epilogues and the whole layer vs the fp32 oracle.

Tolerance (stated once, used everywhere below): operands are bf16/fp16, products
accumulate in fp32, the activated intermediate is stored in the operand dtype and
the output is rounded once to the operand dtype.  Against the pure-fp32 oracle
evaluated on the same rounded operands we require
    max|out - ref| <= 2**-6 * max|ref|      (a few output ulps at the largest magnitude)
    ||out - ref||_F <= 6e-3 * ||ref||_F     (bf16; 1.5e-3 for fp16)
"""
import re
import sys
import tempfile

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _say(msg):
    print("[case] " + msg, flush=True)
    sys.stdout.flush()


def _assert_close(out, ref, dtype, what=""):
    out, ref = out.float().cpu(), ref.float()
    assert torch.isfinite(out).all(), what + ": non-finite output"
    scale = ref.abs().max().clamp(min=1e-30)
    err = (out - ref).abs().max()
    rel_f = (out - ref).norm() / ref.norm().clamp(min=1e-30)
    lim_f = 6e-3 if dtype == torch.bfloat16 else 1.5e-3
    assert err <= 2.0 ** -6 * scale, f"{what}: max abs err {err:.3e} vs scale {scale:.3e}"
    assert rel_f <= lim_f, f"{what}: relative Frobenius error {rel_f:.3e}"


def _inputs(M, H, Fd, E, seed, dtype, zipf=False):
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=seed, zipf=zipf)
    return x.to(dtype), logits, w1.to(dtype), w2.to(dtype)


@pytest.mark.parametrize("M", [1, 16, 64, 200, 512, 2048])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_small_layer_config(native, M, dtype):
    """Small layer (H1024 F3584 E8 top2) at token counts that hit every tile plan."""
    from fast_route_amd import fused_moe
    _say(f"layer C1 M={M} dtype={dtype}")
    x, logits, w1, w2 = _inputs(M, 1024, 3584, 8, 1337, dtype)
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 2, True)
    torch.cuda.synchronize()
    ref = oracle.fused_moe(x, w1, w2, logits, 2, True)
    _assert_close(out, ref, dtype, f"C1 M={M}")


@pytest.mark.parametrize("M", [1, 32, 128, 700])
def test_fine_grained_config(native, M):
    """Fine-grained many-expert shape family (E64 top6, Zipf-skewed load), reduced H/F for CPU oracle time."""
    from fast_route_amd import fused_moe
    _say(f"layer C4-like M={M}")
    x, logits, w1, w2 = _inputs(M, 512, 384, 64, 99, torch.bfloat16, zipf=True)
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 6, True)
    torch.cuda.synchronize()
    ref = oracle.fused_moe(x, w1, w2, logits, 6, True)
    _assert_close(out, ref, torch.bfloat16, f"C4 M={M}")


def test_fine_grained_full_width(native):
    """The fine-grained workload at its real H2048 / F1408 / E64 / top-6 with Zipf-skewed load, every token
    count of its sweep: all tokens against the oracle up to 512, a sample of 48 tokens above."""
    from fast_route_amd import fused_moe
    H, Fd, E, k = 2048, 1408, 64, 6
    _, _, w1, w2 = _inputs(1, H, Fd, E, 5, torch.bfloat16)
    w1d, w2d = w1.cuda(), w2.cuda()
    for M in (1, 32, 128, 512, 2048, 8192):
        _say(f"layer C4 full width M={M}")
        g = torch.Generator().manual_seed(500 + M)
        x = torch.randn(M, H, generator=g).bfloat16()
        logits = oracle.zipf_logits(M, E, 600 + M)
        out = fused_moe(x.cuda(), w1d, w2d, logits.cuda(), k, True)
        torch.cuda.synchronize()
        assert torch.isfinite(out.float()).all()
        sample = torch.arange(M) if M <= 512 else torch.arange(0, M, M // 48)[:48]
        ref = oracle.fused_moe(x[sample], w1, w2, logits[sample], k, True)
        _assert_close(out[sample], ref, torch.bfloat16, f"C4 full M={M}")


def test_layer_edge_cases(native):
    from fast_route_amd import fused_moe, fused_experts
    dtype = torch.bfloat16
    x, logits, w1, w2 = _inputs(96, 256, 128, 8, 3, dtype)
    _say("edge: all tokens to one expert")
    ids = torch.full((96, 1), 5, dtype=torch.int32)
    wts = torch.rand(96, 1)
    out = fused_experts(x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda())
    _assert_close(out, oracle.moe_experts(x, w1, w2, wts, ids), dtype, "one expert")
    _say("edge: topk == E, renormalize False")
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 8, False)
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, 8, False), dtype, "topk==E")
    _say("edge: inplace")
    xd = x.cuda().clone()
    out = fused_moe(xd, w1.cuda(), w2.cuda(), logits.cuda(), 2, True, inplace=True)
    assert out.data_ptr() == xd.data_ptr()
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, 2, True), dtype, "inplace")
    _say("edge: M == 0")
    out = fused_moe(x[:0].cuda(), w1.cuda(), w2.cuda(), logits[:0].cuda(), 2, True)
    assert out.shape == (0, 256)
    _say("edge: int64 ids / fp16 weights accepted by fused_experts")
    w, ids = oracle.gating_topk(logits, 2)
    out = fused_experts(x.cuda(), w1.cuda(), w2.cuda(), w.half().cuda(), ids.long().cuda())
    _assert_close(out, oracle.moe_experts(x, w1, w2, w.half().float(), ids), dtype, "dtype coercion")


@pytest.mark.parametrize("M", [4, 40])
def test_hidden_size_not_multiple_of_long_row_tile(native, M):
    """H = 384 is a multiple of 128 but not of 256: the decode gate/up GEMM must take the
    short-row tile instead of the 512-byte-row one."""
    from fast_route_amd import fused_moe
    _say(f"layer H=384 M={M}")
    x, logits, w1, w2 = _inputs(M, 384, 256, 8, 5, torch.bfloat16)
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 2, True)
    torch.cuda.synchronize()
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, 2, True), torch.bfloat16, f"H=384 M={M}")


def test_token_matrix_of_4gib_is_refused(native):
    """Tile loads address rows by 32-bit byte offsets: a gathered token matrix of 4 GiB
    or more is refused before anything is launched (no memory of that size is touched)."""
    from fast_route_amd import _native as N
    H, Fd, E, k, block = 256, 128, 2, 1, 16
    M = (1 << 32) // (H * 2)  # M*H*2 bytes == 4 GiB exactly
    dummy = torch.zeros(1 << 16, dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    rc = N.lib().fr_moe_gateup_silu(dummy.data_ptr(), dummy.data_ptr(), dummy.data_ptr(), dummy.data_ptr(),
                                    dummy.data_ptr(), M, H, Fd, E, k, block, N.FR_BF16, dummy.data_ptr(), None, st)
    assert rc == -2, rc
    assert b"4 GiB" in N.lib().fr_last_error_string()
    torch.cuda.synchronize()


def test_layer_rejects_bad_arguments(native):
    from fast_route_amd import fused_moe
    x, logits, w1, w2 = _inputs(8, 256, 128, 8, 3, torch.bfloat16)
    with pytest.raises(AssertionError, match="Incompatible dimensions"):
        fused_moe(x[:, :128].contiguous().cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 2)
    with pytest.raises(AssertionError, match="Hidden_states must be contiguous"):
        fused_moe(x.cuda().t().contiguous().t(), w1.cuda(), w2.cuda(), logits.cuda(), 2)
    with pytest.raises(AssertionError):
        fused_moe(x.float().cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 2)
    with pytest.raises(AssertionError):
        fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 9)  # topk > E


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layer_with_64_row_blocks(native, dtype):
    """26 to 52 pairs per expert with H >= 4096: the plan takes 64-row routing blocks (one block per
    expert, K of the down projection cut into slices)."""
    from fast_route_amd import fused_moe
    from fast_route_amd.layers.fused_moe import plan
    _say(f"layer with 64-row blocks {dtype}")
    M, H, Fd, E, k = 160, 4096, 1024, 8, 2
    p = plan(M, H, Fd, E, k, dtype)
    assert p.block == 64 and p.split_k >= 2
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 64, dtype)
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, True)
    torch.cuda.synchronize()
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, "64-row blocks")


@pytest.mark.parametrize("block", [16, 32, 64, 128, 160, 256])
def test_op_level_chain_matches_reference_layer_recipe(native, block):
    """The reference layer spelled with its own ops (layers/stable_route.py:82-102):
    align -> grouped GEMM -> silu_and_mul -> grouped GEMM * weight -> sum."""
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    _say(f"op chain block={block}")
    dtype = torch.bfloat16
    M, H, Fd, E, k = 150, 256, 384, 8, 2
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 21, dtype)
    w, ids = oracle.gating_topk(logits, k)
    xd, w1d, w2d, wd, idd = x.cuda(), w1.cuda(), w2.cuda(), w.cuda(), ids.cuda()
    cfg = {"BLOCK_SIZE_M": block, "BLOCK_SIZE_N": 64, "BLOCK_SIZE_K": 32, "GROUP_SIZE_M": 8}
    s, e, npost = moe_align_block_size(idd, block, E)
    c1 = torch.empty((M, k, 2 * Fd), dtype=dtype, device="cuda")
    invoke_fused_moe_kernel(xd, w1d, c1, wd, idd, s, e, npost, False, k, cfg)
    ref1 = oracle.grouped_gemm(x, w1, w, ids, False, k)
    _assert_close(c1.view(M * k, -1), ref1, dtype, "gemm1")
    c2 = (torch.nn.functional.silu(c1[..., :Fd].float()) * c1[..., Fd:].float()).to(dtype).view(M * k, Fd)
    c3 = torch.empty((M, k, H), dtype=dtype, device="cuda")
    invoke_fused_moe_kernel(c2, w2d, c3, wd, idd, s, e, npost, True, 1, cfg)
    out = c3.float().sum(dim=1)
    torch.cuda.synchronize()
    _assert_close(out, oracle.moe_experts(x, w1, w2, w, ids), dtype, "op chain")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_block_256_several_tiles_per_workgroup(native, dtype):
    """With more 256x256 tiles than resident workgroups the 2-byte kernel walks several
    tiles per workgroup, the next tile's first loads issued during the current tile's last
    K tiles: 27 token blocks x 16 feature tiles = 432 tiles for at most 256 workgroups,
    so the grid mixes workgroups with one tile and with two."""
    from fast_route_amd import fused_moe
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    _say(f"block 256, several tiles per workgroup, {dtype}")
    M, H, Fd, E, k, block = 3000, 512, 2048, 4, 2, 256
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 33, dtype)
    w, ids = oracle.gating_topk(logits, k)
    xd, w1d, w2d, wd, idd = x.cuda(), w1.cuda(), w2.cuda(), w.cuda(), ids.cuda()
    cfg = {"BLOCK_SIZE_M": block, "BLOCK_SIZE_N": 64, "BLOCK_SIZE_K": 32, "GROUP_SIZE_M": 8}
    s, e, npost = moe_align_block_size(idd, block, E)
    c1 = torch.empty((M, k, 2 * Fd), dtype=dtype, device="cuda")
    invoke_fused_moe_kernel(xd, w1d, c1, wd, idd, s, e, npost, False, k, cfg)
    _assert_close(c1.view(M * k, -1), oracle.grouped_gemm(x, w1, w, ids, False, k), dtype, "gemm1")
    c2 = (torch.nn.functional.silu(c1[..., :Fd].float()) * c1[..., Fd:].float()).to(dtype).view(M * k, Fd)
    c3 = torch.empty((M, k, H), dtype=dtype, device="cuda")
    invoke_fused_moe_kernel(c2, w2d, c3, wd, idd, s, e, npost, True, 1, cfg)
    torch.cuda.synchronize()
    _assert_close(c3.float().sum(dim=1), oracle.moe_experts(x, w1, w2, w, ids), dtype, "op chain")
    # the fused layer at the same size takes the same kernels through its own plan
    out = fused_moe(xd, w1d, w2d, logits.cuda(), k, True)
    torch.cuda.synchronize()
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, "layer")


@pytest.mark.parametrize("rows", [256, 160])
@pytest.mark.parametrize("case", ["gate_up_after_whole_tile", "down_first_unit", "with_and_without_scratch"])
def test_last_round_of_tiles_split_along_k(native, rows, case):
    """256-row (and 160-row) tiles that only partly fill the last round of workgroups are cut along K over
    the idle ones and summed by a second launch.  Routing is constructed so that the tile
    counts are exact (k = 1, every expert a whole number of `rows`-token blocks):
    gate_up_after_whole_tile - 17 blocks x 16 feature tiles = 272 tiles, 34 per XCD: one whole
      round of 32 and 2 tiles cut into 8 K slices each (K = 4096 is 64 K tiles);
    down_first_unit - 8 blocks x 2 feature tiles over F = 4096: 2 tiles per XCD in 8 slices
      each, the slice being the workgroup's first and only unit;
    with_and_without_scratch - the two GEMM entry points with and without the scratch agree
      to fp32 summation order (same bf16 result up to one rounding)."""
    from fast_route_amd import _native as N, fused_experts
    from fast_route_amd.layers.fused_moe import plan
    import fast_route_amd as fr
    _say(f"tail split {case} rows={rows}")
    dtype = torch.bfloat16
    if case == "down_first_unit":
        H, Fd, E, blocks = 512, 4096, 2, (5, 3)
    else:
        H, Fd, E, blocks = 4096, 2048, 3, (9, 0, 8)
    M = rows * sum(blocks)
    g = torch.Generator().manual_seed(77)
    x = torch.randn(M, H, generator=g).to(dtype)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.02).to(dtype)
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.02).to(dtype)
    ids = torch.cat([torch.full((rows * b,), e, dtype=torch.int32) for e, b in enumerate(blocks)])
    ids = ids[torch.randperm(M, generator=g)].view(M, 1)
    w = (torch.rand(M, 1, generator=g) + 0.5).float()
    with fr.tunables(block=rows):  # the plan itself keeps a short gate/up K on smaller blocks
        p = plan(M, H, Fd, E, 1, dtype)
    assert p.block == rows and p.tail_bytes > 0 and p.split_k == 1
    xd, w1d, w2d, wd, idd = x.cuda(), w1.cuda(), w2.cuda(), w.cuda(), ids.cuda()
    if case != "with_and_without_scratch":
        with fr.tunables(block=rows):
            out = fused_experts(xd, w1d, w2d, wd, idd)
        torch.cuda.synchronize()
        _assert_close(out, oracle.moe_experts(x, w1, w2, w, ids), dtype, case)
        return
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    lib, st = N.lib(), torch.cuda.current_stream().cuda_stream
    s, e, npost = moe_align_block_size(idd, rows, E)
    tail = torch.empty(p.tail_bytes, dtype=torch.uint8, device="cuda")
    res = []
    for tptr in (None, tail.data_ptr()):
        act = torch.zeros(s.numel(), Fd, dtype=dtype, device="cuda")
        partial = torch.empty(M * H, dtype=torch.float32, device="cuda")
        out = torch.empty(M, H, dtype=dtype, device="cuda")
        N.check(lib.fr_moe_gateup_silu(xd.data_ptr(), w1d.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(), M, H,
                                       Fd, E, 1, rows, N.FR_BF16, act.data_ptr(), tptr, st))
        N.check(lib.fr_moe_down_combine(act.data_ptr(), w2d.data_ptr(), wd.data_ptr(), s.data_ptr(), e.data_ptr(),
                                        npost.data_ptr(), M, H, Fd, E, 1, rows, 1, N.FR_BF16, partial.data_ptr(),
                                        out.data_ptr(), tptr, st))
        torch.cuda.synchronize()
        res.append((act.float().cpu(), out.float().cpu()))
    (act0, out0), (act1, out1) = res
    assert not torch.equal(act0, act1), "the scratch changed nothing: the split path did not run"
    # one bf16 rounding apart at most (2^-8 relative), on values whose fp32 sums differ in the last bits
    assert ((act0 - act1).abs() <= 2.0 ** -7 * act0.abs().clamp(min=1e-3)).all()
    assert ((out0 - out1).abs() <= 2.0 ** -6 * out0.abs().max()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,H,E,k", [(1, 4096, 8, 2), (2, 4096, 8, 2), (3, 4096, 8, 2), (4, 4096, 8, 2), (4, 8192, 4, 2),
                                      (2, 4096, 16, 6), (1, 8192, 8, 8), (3, 5120, 4, 2), (2, 6144, 8, 2), (4, 7168, 4, 3)])
def test_decode_gate_up_by_rows(native, M, H, E, k, dtype):
    """Up to four tokens with H = 4096, 5120, 6144, 7168 or 8192 (rows of 5 to 8 rounds' chunks): the gate/up
    projection streams each weight row
    past the routing block's token rows (dot products, no tiles) and leaves the same activation
    layout to the down projection.  H = 8192 with four tokens fills the token-row buffer."""
    from fast_route_amd import fused_moe
    _say(f"decode rows M={M} H={H} E={E} k={k} {dtype}")
    x, logits, w1, w2 = _inputs(M, H, 384, E, 100 + M + k, dtype)
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, True)
    torch.cuda.synchronize()
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, f"rows M={M} H={H}")


@pytest.mark.parametrize("block", [16, 32, 64, 128])
def test_decode_gate_up_by_rows_matches_tiles(native, block):
    """The same three tokens through the gate/up entry point with H = 4096 (rows, for blocks up to
    64 slots; 128-slot blocks keep the tiles) and, zero-extended to H = 4224 (not a multiple of
    4096: tiles), give the same activations up to the summation order; an expert chosen twice by
    one token puts more rows into a block than there are tokens, which costs the row form a second
    pass over that block."""
    from fast_route_amd import _native as N
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    _say(f"decode rows vs tiles block={block}")
    dtype = torch.bfloat16
    M, H, Fd, E, k = 3, 4096, 256, 4, 2
    g = torch.Generator().manual_seed(block)
    x = torch.randn(M, H, generator=g).to(dtype)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.02).to(dtype)
    ids = torch.tensor([[1, 1], [1, 3], [0, 1]], dtype=torch.int32)   # expert 1: 4 rows from 3 tokens
    lib, st = N.lib(), torch.cuda.current_stream().cuda_stream
    s, e, npost = moe_align_block_size(ids.cuda(), block, E)
    acts = []
    for pad in (0, 128):
        xd = torch.nn.functional.pad(x, (0, pad)).contiguous().cuda()
        w1d = torch.nn.functional.pad(w1, (0, pad)).contiguous().cuda()
        act = torch.zeros(s.numel(), Fd, dtype=dtype, device="cuda")
        N.check(lib.fr_moe_gateup_silu(xd.data_ptr(), w1d.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(), M,
                                       H + pad, Fd, E, k, block, N.FR_BF16, act.data_ptr(), None, st))
        torch.cuda.synchronize()
        acts.append(act.float().cpu())
    # reference: every real slot's row (the tile kernel also fills the padding slots of a block, with
    # values nobody reads; the row form leaves them alone)
    sc = s.cpu()
    ref = torch.zeros_like(acts[0])
    real = torch.zeros(ref.shape[0], dtype=torch.bool)
    for slot in range(int(npost.item())):
        sid = int(sc[slot])
        if sid < M * k:
            gu = x[sid // k].float() @ w1[int(ids.view(-1)[sid])].float().T
            ref[slot] = torch.nn.functional.silu(gu[:Fd]) * gu[Fd:]
            real[slot] = True
    assert int(real.sum()) == M * k
    for a in acts:
        assert ((a - ref).abs() <= 2.0 ** -7 * ref.abs() + 1e-3)[real].all()
    if block <= 64:
        assert acts[0][~real].abs().sum() == 0


@pytest.mark.parametrize("M", [2, 16, 1536])
def test_layer_under_graph_capture(native, M):
    """The whole layer (router logits form) captured into a HIP graph after one warm-up call and
    replayed three times, with eager work and synchronisations between the replays and new inputs
    written into the captured buffers: every replay equals the eager result bit for bit.  M=2
    (with H = 4096) takes the gate/up projection by weight rows, M=16
    takes the decode kernels and the fused route+align launch, M=1536 the persistent kernels with
    their split last round and fix-up launches."""
    from fast_route_amd import _native as N
    from fast_route_amd.layers.fused_moe import plan
    _say(f"graph capture M={M}")
    dtype = torch.bfloat16
    H, Fd, E, k = (4096, 512, 4, 2) if M == 2 else (1024, 2048, 4, 2)
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 55, dtype)
    xd, ld, w1d, w2d = x.cuda(), logits.cuda(), w1.cuda(), w2.cuda()
    p = plan(M, H, Fd, E, k, dtype)
    ws = torch.empty(max(p.workspace_bytes, 256), dtype=torch.uint8, device="cuda")
    out = torch.empty(M, H, dtype=dtype, device="cuda")
    lib = N.lib()

    def call(stream):
        N.check(lib.fr_fused_moe(xd.data_ptr(), w1d.data_ptr(), w2d.data_ptr(), ld.data_ptr(), N.FR_F32, M, H, Fd, E, k, 1,
                                 N.FR_BF16, out.data_ptr(), ws.data_ptr(), ws.numel(), stream))

    call(torch.cuda.current_stream().cuda_stream)  # warm-up: per-kernel attributes are set on first use
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call(torch.cuda.current_stream().cuda_stream)
    for rep in range(3):
        gen = torch.Generator().manual_seed(100 + rep)
        xd.copy_(torch.randn(M, H, generator=gen).to(dtype))
        ld.copy_(torch.randn(M, E, generator=gen))
        call(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        eager = out.clone()
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from the eager result"
    _assert_close(out, oracle.fused_moe(xd.cpu(), w1, w2, ld.cpu(), k, True), dtype, "graph replay")


@pytest.mark.parametrize("block", [128, 160, 256])
def test_grouped_gemm_with_blocks_in_any_order(native, block):
    """The op-level GEMM only needs every block to belong to one expert; routing arrays whose
    blocks are not in ascending expert order (here: reversed) are legal input.  The persistent
    kernels walk tiles expert by expert through a table built from an ascending expert_ids and
    must fall back to a plain walk when it is not."""
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    _say(f"grouped GEMM, blocks reversed, block={block}")
    dtype = torch.bfloat16
    M, H, Fd, E, k = 1200, 512, 768, 6, 2
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 41, dtype)
    w, ids = oracle.gating_topk(logits, k)
    xd, w1d, wd, idd = x.cuda(), w1.cuda(), w.cuda(), ids.cuda()
    s, e, npost = moe_align_block_size(idd, block, E)
    nb = int(npost.item()) // block
    s2, e2 = s.clone(), e.clone()
    s2[: nb * block] = s[: nb * block].view(nb, block).flip(0).reshape(-1)
    e2[:nb] = e[:nb].flip(0)
    cfg = {"BLOCK_SIZE_M": block, "BLOCK_SIZE_N": 64, "BLOCK_SIZE_K": 32, "GROUP_SIZE_M": 8}
    c1 = torch.empty((M, k, 2 * Fd), dtype=dtype, device="cuda")
    invoke_fused_moe_kernel(xd, w1d, c1, wd, idd, s2, e2, npost, False, k, cfg)
    torch.cuda.synchronize()
    _assert_close(c1.view(M * k, -1), oracle.grouped_gemm(x, w1, w, ids, False, k), dtype, "reversed blocks")


@pytest.mark.parametrize("block", [32, 64, 128, 160, 256])
@pytest.mark.parametrize("E", [3, 70, 300])
def test_grouped_gemm_with_pairs_anywhere_in_their_block(native, block, E):
    """Routing arrays of another producer: pairs and padding of a block in any order, a run's last block with one pair in
    its last slot, more experts than a workgroup has threads for, experts without a block."""
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel
    _say(f"grouped GEMM, shuffled blocks, block={block} E={E}")
    dtype, K, N = torch.bfloat16, 1024, 256
    rng = np.random.default_rng(E + block)
    counts = rng.integers(0, 2 * block + 1, E) * (rng.random(E) < 40 / (E + 20))
    counts[E // 2] = block + 1
    n = int(counts.sum())
    pairs = rng.permutation(n)
    s, e, at = [], [], 0
    for x in range(E):
        left = pairs[at : at + counts[x]]
        at += counts[x]
        while len(left):
            b = np.full(block, n)
            take = left[: 1 if x == E // 2 and len(left) == counts[x] else block]
            left = left[len(take):]
            b[[block - 1] if len(take) == 1 else rng.choice(block, len(take), replace=False)] = take
            s.append(b)
            e.append(x)
    a = torch.randn(n, K, generator=torch.Generator().manual_seed(E)).to(dtype)
    w = (torch.randn(E, N, K, generator=torch.Generator().manual_seed(block)) * 0.02).to(dtype)
    sid, eid = torch.from_numpy(np.concatenate(s)).int().cuda(), torch.tensor(e, dtype=torch.int32, device="cuda")
    npost = torch.tensor([len(e) * block], dtype=torch.int32, device="cuda")
    ids = torch.empty(n, 1, dtype=torch.int32)
    ids[torch.from_numpy(pairs).long(), 0] = torch.from_numpy(np.repeat(np.arange(E), counts)).int()
    c = torch.zeros(n, 1, N, dtype=dtype, device="cuda")
    cfg = {"BLOCK_SIZE_M": block, "BLOCK_SIZE_N": 64, "BLOCK_SIZE_K": 32, "GROUP_SIZE_M": 8}
    wt = torch.ones(n, 1)
    invoke_fused_moe_kernel(a.cuda(), w.cuda(), c, wt.cuda(), ids.cuda(), sid, eid, npost, False, 1, cfg)
    torch.cuda.synchronize()
    _assert_close(c.view(n, N), oracle.grouped_gemm(a, w, wt, ids, False, 1), dtype, "pairs anywhere")


@pytest.mark.parametrize("N", [256, 260, 388, 516])
@pytest.mark.parametrize("block", [16, 32, 64, 128, 160, 256])
def test_rows_of_whole_and_partial_tiles(native, block, N):
    """16-byte stores of whole tiles: output rows that start at multiples of 8 bytes only (N = 4 mod 8), with a last tile that is
    narrower than the others; K long enough for the 256-row tile with one wavefront per SIMD.  What lies around C stays as it is."""
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    _say(f"grouped GEMM, N={N}, block={block}")
    M, K, E, k = 300, 1024, 5, 2
    for dtype in (torch.bfloat16, torch.float16):
        x, logits, _, w = _inputs(M, N, K, E, 43 + N, dtype)  # w: [E, N, K]
        x = torch.randn(M, K, generator=torch.Generator().manual_seed(N)).to(dtype)
        wt, ids = oracle.gating_topk(logits, k)
        s, e, npost = moe_align_block_size(ids.cuda(), block, E)
        cfg = {"BLOCK_SIZE_M": block, "BLOCK_SIZE_N": 64, "BLOCK_SIZE_K": 32, "GROUP_SIZE_M": 8}
        guard = 8 * N
        buf = torch.full((2 * guard + M * k * N,), 7.0, dtype=dtype, device="cuda")
        c = buf[guard:-guard].view(M, k, N)
        invoke_fused_moe_kernel(x.cuda(), w.cuda(), c, wt.cuda(), ids.cuda(), s, e, npost, True, k, cfg)
        torch.cuda.synchronize()
        assert (buf[:guard] == 7).all() and (buf[-guard:] == 7).all()
        _assert_close(c.view(M * k, N), oracle.grouped_gemm(x, w, wt, ids, True, k), dtype, f"{dtype}")


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("H,Fd", [(384, 1152), (640, 1664), (2048, 1152), (2432, 2176), (384, 2048)])
@pytest.mark.parametrize("block", [16, 32, 64, 128, 160])
def test_k_starts_of_tiles_alone_on_their_weights(native, block, H, Fd, split):
    """A tile that is alone on its weight tile (16 and 32 rows: any tile) walks its K tiles from a place of its own, round the end:
    K loops from the shortest the persistent kernels take (6 K tiles) up, odd counts, K slices and cut last rounds, experts with one
    block next to experts with several and with none; gate/up rows on both sides of 4 KB (2048 elements: the last of the short ones), where
    32 and 64 rows have forms of their own, and 64-row down projections with fewer tiles than CUs (one slice) and with more (three)."""
    import fast_route_amd as fr
    from fast_route_amd import fused_experts
    E = 12
    counts = np.array([block, block - 1, 1, 0, 17, 3 * block + 5, block // 2, 0, block + 1, 33, 2, block])
    rng = np.random.default_rng(H + block)
    ids = torch.from_numpy(rng.permutation(np.repeat(np.arange(E), counts))).int().view(-1, 1)
    M = ids.shape[0]
    _say(f"K starts block={block} H={H} F={Fd} split={split}")
    for dtype in (torch.bfloat16, torch.float16):
        x, _, w1, w2 = _inputs(M, H, Fd, E, 5 + H, dtype)
        wts = torch.rand(M, 1, generator=torch.Generator().manual_seed(M)) + 0.5
        ref = oracle.moe_experts(x, w1, w2, wts, ids)
        xd, w1d, w2d, wd, idd = x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda()
        try:
            with fr.tunables(block=block, split_k=split, no_quad=True):
                out, again = fused_experts(xd, w1d, w2d, wd, idd), fused_experts(xd, w1d, w2d, wd, idd)
        finally:
            fr.reset_tunables()
        torch.cuda.synchronize()
        assert torch.equal(out, again)
        _assert_close(out, ref, dtype, f"{dtype}")


@pytest.mark.parametrize("H,form", [(640, "32, 128, 128"), (1152, "32, 128, 128"), (1024, "32, 64, 256"), (2048, "32, 64, 256"), (2304, "32, 128, 512"), (2176, "32, 128, 128")])
def test_gate_up_forms_of_32_rows(native, kernels_of, H, form):
    """Weight rows of up to 4 KB take the narrow 32-row tile only where whole 512-byte pieces make them up."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    M, Fd, E, k = 100, 1024, 8, 2
    _say(f"32-row gate/up H={H}")
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 7 + H, torch.bfloat16)
    try:
        with fr.tunables(block=32):
            out, names = kernels_of(lambda: fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, True))
    finally:
        fr.reset_tunables()
    gate_up = [n for n in names if "moe_gemm" in n and re.search(r"Li1EEEv|, 1>\(", n)]  # EPI_SILU
    mangled = "CfgILi" + form.replace(", ", "ELi") + "E"
    assert len(gate_up) == 1 and (mangled in gate_up[0] or "Cfg<" + form + "," in gate_up[0]), names
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), torch.bfloat16, "layer")


@pytest.mark.parametrize("Fd,split,slots", [(8192, 1, 2), (8192, 2, 3), (8064, 1, 3), (8320, 1, 3), (16384, 2, 2), (1408, 1, 3), (4096, 1, 3)])
def test_ring_slots_of_the_32_row_down_projection(native, kernels_of, Fd, split, slots):
    """Two ring slots only for K slices of 16 KB or more of weight rows a power of two long, three otherwise."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    M, H, E, k = 100, 384, 8, 2
    _say(f"32-row down projection F={Fd} split={split}")
    for dtype in (torch.bfloat16, torch.float16):
        x, logits, w1, w2 = _inputs(M, H, Fd, E, 9 + Fd, dtype)
        try:
            with fr.tunables(block=32, split_k=split):
                out, names = kernels_of(lambda: fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, True))
        finally:
            fr.reset_tunables()
        down = [n for n in names if "moe_gemm" in n and not re.search(r"Li1EEEv|, 1>\(", n)]
        assert len(down) == 1 and re.search(r"ILi32ELi128ELi128ELi1ELi4ELi16ELi2ELi%dE|<32, 128, 128, 1, 4, 16, 2, %d," % (slots, slots), down[0]), names
        _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, f"{dtype}")


@pytest.mark.parametrize("Fd,H,slots", [(128, 2048, 4), (256, 2048, 4), (384, 2048, 4), (512, 2048, 4), (1408, 2048, 4), (2048, 2048, 4), (2176, 2048, 3), (512, 512, 3)])
def test_four_ring_slots_of_short_down_projections(native, kernels_of, Fd, H, slots):
    """32-row down projection, weight rows of up to 4 KB in a launch of 512 tiles or more by the worst-case count: four ring slots, with
    fewer K tiles than slots, as many, and more; three for longer rows and for fewer tiles.  Reference: float32 on the operands."""
    from fast_route_amd import fused_moe
    M, E, k = 64, 32, 4
    _say(f"slots of the 32-row down projection F={Fd} H={H}")
    for dtype in (torch.bfloat16, torch.float16):
        g = torch.Generator(device="cuda").manual_seed(11 + Fd)
        x = torch.randn(M, H, generator=g, device="cuda").to(dtype)
        w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).to(dtype)
        w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).to(dtype)
        logits = torch.randn(M, E, generator=g, device="cuda")
        import fast_route_amd as fr
        with fr.tunables(block=32, split_k=1):
            out, names = kernels_of(lambda: fused_moe(x, w1, w2, logits, k, True))
        down = [n for n in names if "moe_gemm" in n and not re.search(r"Li1EEEv|, 1>\(", n)]
        assert len(down) == 1 and re.search(r"ILi32ELi128ELi128ELi1ELi4ELi16ELi2ELi%dE|<32, 128, 128, 1, 4, 16, 2, %d," % (slots, slots), down[0]), names
        top, ids = torch.topk(logits, k, dim=1)
        weights, ref = torch.softmax(top, dim=1), torch.zeros(M, H, device="cuda")
        for e in range(E):
            token, slot = (ids == e).nonzero(as_tuple=True)
            gate, up = (x[token].float() @ w1[e].float().t()).chunk(2, dim=1)
            ref.index_add_(0, token, ((torch.nn.functional.silu(gate) * up) @ w2[e].float().t()) * weights[token, slot][:, None])
        _assert_close(out, ref.cpu(), dtype, f"{dtype}")


@pytest.mark.parametrize("Fd,slots", [(4096, 4), (4352, 3)])
def test_four_ring_slots_of_split_down_projections(native, kernels_of, Fd, slots):
    """Two K slices of longer weight rows: four ring slots up to 4 KB of a slice, three beyond.  Reference: float32 on the operands."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    M, E, k, H = 64, 32, 4, 1024
    _say(f"slots of a split 32-row down projection F={Fd}")
    for dtype in (torch.bfloat16, torch.float16):
        g = torch.Generator(device="cuda").manual_seed(17 + Fd)
        x = torch.randn(M, H, generator=g, device="cuda").to(dtype)
        w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).to(dtype)
        w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).to(dtype)
        logits = torch.randn(M, E, generator=g, device="cuda")
        with fr.tunables(block=32, split_k=2):
            out, names = kernels_of(lambda: fused_moe(x, w1, w2, logits, k, True))
        down = [n for n in names if "moe_gemm" in n and not re.search(r"Li1EEEv|, 1>\(", n)]
        assert len(down) == 1 and re.search(r"ILi32ELi128ELi128ELi1ELi4ELi16ELi2ELi%dE|<32, 128, 128, 1, 4, 16, 2, %d," % (slots, slots), down[0]), names
        top, ids = torch.topk(logits, k, dim=1)
        weights, ref = torch.softmax(top, dim=1), torch.zeros(M, H, device="cuda")
        for e in range(E):
            token, slot = (ids == e).nonzero(as_tuple=True)
            gate, up = (x[token].float() @ w1[e].float().t()).chunk(2, dim=1)
            ref.index_add_(0, token, ((torch.nn.functional.silu(gate) * up) @ w2[e].float().t()) * weights[token, slot][:, None])
        _assert_close(out, ref.cpu(), dtype, f"{dtype}")


def test_stable_and_vllm_route_layers(native):
    """Gate-matrix entry points of both reference layers."""
    from fast_route_amd.layers import stable_route, vllm_route
    _say("gate-matrix layers")
    dtype = torch.bfloat16
    M, H, Fd, E, k = 80, 512, 256, 16, 2
    x, _, w1, w2 = _inputs(M, H, Fd, E, 8, dtype)
    gate = (torch.randn(H, E, generator=torch.Generator().manual_seed(1)) / 8).to(dtype)
    a = stable_route.fused_moe(x.cuda(), gate.cuda(), w1.cuda(), w2.cuda(), k, True)
    b = vllm_route.fused_moe(x.cuda(), gate.cuda(), w1.cuda(), w2.cuda(), k, True)
    torch.cuda.synchronize()
    # routing decided from fp32 logits on device; take the device's own selection for the oracle
    from fast_route_amd.ops.stable_route import fused_route
    tw = torch.empty(M, k, dtype=torch.float32, device="cuda")
    ti = torch.empty(M, k, dtype=torch.int32, device="cuda")
    w, ids = fused_route(x.cuda(), gate.cuda(), k, tw, ti, True)
    ref = oracle.moe_experts(x, w1, w2, w.cpu(), ids.cpu())
    _assert_close(a, ref, dtype, "stable_route layer")
    # the baseline layer rounds logits to bf16 before gating: compare on tokens routed identically
    lw, lid = oracle.gating_topk(torch.matmul(x.cuda(), gate.cuda()).cpu(), k, True)
    same = (lid == ids.cpu()).all(dim=1)
    assert same.float().mean() > 0.8
    refb = oracle.moe_experts(x, w1, w2, lw, lid)
    _assert_close(b, refb, dtype, "vllm_route layer")


def test_profile_twin_matches_layer_and_writes_trace(native, tmp_path):
    """layers/profile_fused_route.py: same result as the fused layer, bit for bit (same
    kernels, same plan), and a chrome trace with one complete event per stage."""
    import json
    from fast_route_amd.layers import profile_fused_route, stable_route
    _say("profile twin")
    dtype = torch.bfloat16
    M, H, Fd, E, k = 96, 512, 256, 8, 2
    x, _, w1, w2 = _inputs(M, H, Fd, E, 12, dtype)
    gate = (torch.randn(H, E, generator=torch.Generator().manual_seed(2)) / 8).to(dtype)
    ref = stable_route.fused_moe(x.cuda(), gate.cuda(), w1.cuda(), w2.cuda(), k, True)
    out = profile_fused_route.fused_moe(x.cuda(), gate.cuda(), w1.cuda(), w2.cuda(), k, True, save_dir=str(tmp_path))
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    # and against the oracle: routing from fp64 logits; tokens whose fp32 near-tie flipped an id are left out
    ow, oid = oracle.route_from_gate(x, gate, k)
    from fast_route_amd.ops.stable_route import fused_route
    tw = torch.empty(M, k, dtype=torch.float32, device="cuda")
    ti = torch.empty(M, k, dtype=torch.int32, device="cuda")
    _, ids = fused_route(x.cuda(), gate.cuda(), k, tw, ti, True)
    same = (ids.cpu() == oid).all(dim=1)
    assert same.float().mean() > 0.95
    want = oracle.moe_experts(x, w1, w2, ow, oid)
    _assert_close(out[same.cuda()], want[same], dtype, "profile twin vs oracle")
    path = tmp_path / f"fused_breakdown_{M}_{H}_{E}_{2 * Fd}_{k}.json"
    trace = json.loads(path.read_text())
    names = [e["name"] for e in trace["traceEvents"]]
    assert names == list(profile_fused_route.STAGES)
    assert all(e["ph"] == "X" and e["dur"] > 0 for e in trace["traceEvents"])
    ts = [e["ts"] for e in trace["traceEvents"]]
    assert ts == sorted(ts)


def test_transformer_layer_bench_runs_and_matches_its_parts(native):
    """fast_route_amd.transformer_layer_bench: the layer is attention + residual + the
    gate-matrix MoE; its output equals the MoE entry point applied to attn(x) + x."""
    from fast_route_amd import transformer_layer_bench as tb
    from fast_route_amd.layers.stable_route import fused_moe
    _say("transformer layer bench")
    rec, out, (gate, w1, w2, attn) = tb.run(seq=64, n=256, k=512, e=8, topk=2, b=2, n_head=4, head_dim=64,
                                            reps=3, warmup=1)
    assert out.shape == (2 * 64, 512) and torch.isfinite(out.float()).all()
    assert 0.0 < rec["moe_share"] <= 1.0 and rec["layer_ms"] > 0 and rec["layer_ms_p20"] <= rec["layer_ms_p80"]
    g = torch.Generator(device="cuda").manual_seed(1337)
    x = torch.randn((2, 64, 512), device="cuda", dtype=torch.float16, generator=g) / 10
    with torch.no_grad():
        h = (attn(x) + x).view(-1, 512)
        again = fused_moe(h, gate, w1, w2, 2, True, False)
    assert torch.equal(out, again)
    # against the oracle: the MoE of the layer's own attention output, routed and multiplied on the CPU
    hc, gc = h.cpu(), gate.cpu()
    ow, oid = oracle.route_from_gate(hc, gc, 2)
    from fast_route_amd.ops.stable_route import fused_route
    tw = torch.empty(h.shape[0], 2, dtype=torch.float32, device="cuda")
    ti = torch.empty(h.shape[0], 2, dtype=torch.int32, device="cuda")
    _, ids = fused_route(h, gate, 2, tw, ti, True)
    same = (ids.cpu() == oid).all(dim=1)
    assert same.float().mean() > 0.95
    want = oracle.moe_experts(hc, w1.cpu(), w2.cpu(), ow, oid)
    _assert_close(out[same.cuda()], want[same], torch.float16, "transformer layer vs oracle")


def test_mixtral_shape_sampled_tokens_and_properties(native):
    """Mixtral-8x7B shape at full size (H4096 F14336 E8 top2), every token count of its sweep:
    oracle on a sample of tokens and determinism; at 16 and 4096 tokens also the size-independent
    properties (batch independence, linearity in the routed weights) on all tokens."""
    from fast_route_amd import fused_moe, fused_experts
    dtype = torch.bfloat16
    H, Fd, E, k = 4096, 14336, 8, 2
    g = torch.Generator(device="cuda").manual_seed(1337)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).to(dtype)
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).to(dtype)
    w1c, w2c = w1.cpu(), w2.cpu()
    for M in (1, 16, 64, 256, 1024, 4096, 16384):
        _say(f"mixtral full width M={M}")
        x = torch.randn(M, H, generator=g, device="cuda").to(dtype)
        logits = torch.randn(M, E, generator=g, device="cuda")
        out = fused_moe(x, w1, w2, logits, k, True)
        torch.cuda.synchronize()
        assert torch.isfinite(out.float()).all()
        sample = torch.arange(0, M, max(1, M // 24))[:24]
        ref = oracle.fused_moe(x[sample].cpu(), w1c, w2c, logits[sample].cpu(), k, True)
        _assert_close(out[sample], ref, dtype, f"mixtral M={M} sample")
        # determinism: same call, same bits
        out2 = fused_moe(x, w1, w2, logits, k, True)
        assert torch.equal(out, out2)
        if M not in (16, 4096):
            continue
        # a token's output does not depend on which other tokens share the batch
        half = fused_moe(x[: M // 2].contiguous(), w1, w2, logits[: M // 2].contiguous(), k, True)
        _assert_close(half, out[: M // 2].float().cpu(), dtype, "batch independence")
        # linearity in the routed weights: doubling them doubles the output (exact in binary fp)
        from fast_route_amd.ops.stable_route import topk_softmax
        w = torch.empty((M, k), dtype=torch.float32, device="cuda")
        ids = torch.empty((M, k), dtype=torch.int32, device="cuda")
        topk_softmax(w, ids, None, logits, renormalize=True)
        a = fused_experts(x, w1, w2, w, ids)
        b = fused_experts(x, w1, w2, 2 * w, ids)
        assert torch.equal(a, out) and torch.equal(b.float(), 2 * a.float())


@pytest.mark.parametrize("m", [1, 33, 222, 1024])
def test_reference_end_to_end_recipe(native, m):
    """The reference's own end-to-end check replayed (benchmarks/swizzle_moe/perf_test_moe.py:34-73):
    fp16 operands drawn as randn / 10, routing = torch.topk(softmax(randn score)), no renormalisation,
    experts-only entry point, torch_moe as the expectation, assert_close(atol=1e-2, rtol=0).
    Widths are scaled down from the reference's n=14336 / k=4096 to keep the CPU expectation quick."""
    from fast_route_amd import fused_experts
    n, k, e, topk = 1024, 512, 8, 2
    _say(f"reference recipe m={m} n={n} k={k} e={e} topk={topk}")
    torch.manual_seed(3227)  # the reference's seed for this check
    a = (torch.randn((m, k)) / 10).half()
    w1 = (torch.randn((e, 2 * n, k)) / 10).half()
    w2 = (torch.randn((e, k, n)) / 10).half()
    score = torch.softmax(torch.randn((m, e)), dim=-1)
    topk_weight, topk_ids = torch.topk(score, topk)
    out = fused_experts(a.cuda(), w1.cuda(), w2.cuda(), topk_weight.cuda(), topk_ids.cuda(), inplace=False)
    torch.cuda.synchronize()
    want = oracle.moe_experts(a, w1, w2, topk_weight, topk_ids)
    torch.testing.assert_close(out.float().cpu(), want, atol=1e-2, rtol=0)


@pytest.mark.parametrize("E,k,H,Fd", [(8, 2, 256, 4096), (8, 2, 512, 5120), (16, 6, 256, 4096), (8, 8, 128, 8192),
                                      (4, 1, 384, 14336), (64, 6, 256, 16384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_down_projection_by_rows(native, E, k, H, Fd, dtype):
    """At most 4 routed pairs and weight rows of 4096..16384 elements (multiples of 512): the down
    projection streams weight rows past the activated rows and sums a token's pairs itself - no partial
    buffer, no combine launch.  Token counts on both sides of that limit (up to 8 pairs), against the
    oracle; the same bits on every run."""
    from fast_route_amd import fused_moe, fused_experts
    for M in range(1, 8 // k + 1):
        _say(f"down by rows E={E} k={k} H={H} F={Fd} {dtype} M={M}")
        x, logits, w1, w2 = _inputs(M, H, Fd, E, 77 + M, dtype)
        xd, w1d, w2d, ld = x.cuda(), w1.cuda(), w2.cuda(), logits.cuda()
        out = fused_moe(xd, w1d, w2d, ld, k, True)
        torch.cuda.synchronize()
        _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, f"down by rows M={M}")
        for _ in range(3):
            assert torch.equal(fused_moe(xd, w1d, w2d, ld, k, True), out)
    if k == 2 and E >= 4:
        _say("down by rows: a token naming one expert twice, another token sharing it")
        ids = torch.tensor([[3, 3], [3, 1], [0, 2]], dtype=torch.int32)
        wts = torch.tensor([[0.25, 0.5], [0.7, 0.3], [0.9, 0.1]])
        x, _, w1, w2 = _inputs(3, H, Fd, E, 5, dtype)
        out = fused_experts(x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda())
        _assert_close(out, oracle.moe_experts(x, w1, w2, wts, ids), dtype, "down by rows, repeated expert")


def test_tunables_and_prepare(native):
    """Plan overrides (routing block, K slices, walk group, no last-round split) change the kernels a layer takes,
    never its result beyond fp32 summation order; fr_moe_prepare sets every kernel up without launching."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    dtype = torch.bfloat16
    fr.prepare(dtype)
    fr.prepare(torch.float16)
    fr.prepare("fp8")
    torch.cuda.synchronize()
    x, logits, w1, w2 = _inputs(300, 512, 1024, 8, 21, dtype)
    xd, w1d, w2d, ld = x.cuda(), w1.cuda(), w2.cuda(), logits.cuda()
    ref = oracle.fused_moe(x, w1, w2, logits, 2, True)
    base = fused_moe(xd, w1d, w2d, ld, 2, True)
    _assert_close(base, ref, dtype, "library plan")
    try:
        for kw in ({"block": 16}, {"block": 32, "split_k": 3}, {"block": 64, "group_m": 1}, {"block": 128, "split_k": 2},
                   {"block": 256, "no_tail_split": True}, {"block": 256, "group_m": 3}, {"split_k": 4}, {"group_m": 64},
                   {"block": 160}, {"block": 160, "split_k": 2}):
            _say(f"tunables {kw}")
            with fr.tunables(**kw):
                out = fused_moe(xd, w1d, w2d, ld, 2, True)
            torch.cuda.synchronize()
            _assert_close(out, ref, dtype, f"tunables {kw}")
            assert (out.float() - base.float()).abs().max() <= 2.0 ** -7 * ref.abs().max()
    finally:
        fr.reset_tunables()
    assert torch.equal(fused_moe(xd, w1d, w2d, ld, 2, True), base)


@pytest.mark.parametrize("block,kind", [(128, "bf16"), (160, "bf16"), (256, "bf16"), (128, "fp8"), (160, "fp8"), (256, "fp8")])
def test_persistent_tiles_alternating_half_empty_and_full_blocks(native, block, kind):
    """The persistent 128-, 160- and 256-row kernels let the wavefronts of a block's upper half skip their fragment
    reads and MFMAs when that half holds only padding, and pick the fragments up again when their next block
    has rows.  64 experts with one routing block each, a seeded mix of full blocks and blocks filled to less
    than half, 8 feature tiles per block: every workgroup walks several units and meets both transitions."""
    import fast_route_amd as fr
    from fast_route_amd import fused_experts, fused_moe_fp8, prepare_weights_fp8
    E, H, Fd = 64, 512, 1024
    if (block, kind) == (160, "fp8"):
        H = 1024  # that tile has no plain form: five K tiles of 128 bytes per K slice at least
    rng = np.random.default_rng(block)
    counts = np.where(rng.random(E) < 0.5, block, rng.integers(1, block // 2 + 1, E))
    ids = torch.from_numpy(np.repeat(np.arange(E), counts)).int()
    ids = ids[torch.from_numpy(rng.permutation(ids.numel()))].view(-1, 1)
    M = ids.shape[0]
    _say(f"persistent half/full blocks block={block} {kind} M={M}")
    x, _, w1, w2 = _inputs(M, H, Fd, E, 31 + block, torch.bfloat16)
    try:
        with fr.tunables(block=block):
            if kind == "bf16":
                wts = torch.rand(M, 1) + 0.5
                out = fused_experts(x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda())
                torch.cuda.synchronize()
                _assert_close(out, oracle.moe_experts(x, w1, w2, wts, ids), torch.bfloat16, "half/full blocks")
            else:
                logits = torch.full((M, E), -20.0)
                logits[torch.arange(M), ids.view(-1).long()] = 20.0
                w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
                out = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), 1, True)
                torch.cuda.synchronize()
                ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, 1, True)
                o = out.float().cpu()
                assert torch.isfinite(o).all()
                assert (o - ref).norm() / ref.norm() <= 1e-2 and (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()
    finally:
        fr.reset_tunables()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_wavefront_per_simd_tile_equals_the_eight_wavefront_tile(native, dtype):
    """256-row blocks with 16 K tiles or more run on four wavefronts of 128 x 128 outputs (moe_gemm_quad_kernel);
    the no_quad knob sends the same call to the eight-wavefront kernel.  Same MFMA shape and K order: outputs equal
    bit for bit, and both match the oracle.  64 experts with a seeded mix of full, under-half and over-half blocks,
    16 / 8 feature tiles: every workgroup walks several units (hand-over of the ring), meets all-padding halves,
    and the last round of tiles is split along K (32 K tiles in the gate/up GEMM)."""
    import fast_route_amd as fr
    from fast_route_amd import fused_experts, fused_moe
    E, H, Fd = 64, 2048, 2048
    rng = np.random.default_rng(5)
    counts = np.where(rng.random(E) < 0.4, 256, rng.integers(1, 200, E))
    ids = torch.from_numpy(np.repeat(np.arange(E), counts)).int()
    ids = ids[torch.from_numpy(rng.permutation(ids.numel()))].view(-1, 1)
    M = ids.shape[0]
    _say(f"quad tile vs eight-wavefront tile {dtype} M={M}")
    x, _, w1, w2 = _inputs(M, H, Fd, E, 77, dtype)
    wts = torch.rand(M, 1) + 0.5
    xd, w1d, w2d, wd, idd = x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda()
    try:
        with fr.tunables(block=256):
            quad = fused_experts(xd, w1d, w2d, wd, idd)
        with fr.tunables(block=256, no_quad=True):
            eight = fused_experts(xd, w1d, w2d, wd, idd)
        with fr.tunables(block=256, no_tail_split=True):
            whole = fused_experts(xd, w1d, w2d, wd, idd)
        torch.cuda.synchronize()
        assert torch.equal(quad, eight), "the two 256-row kernels differ"
        _assert_close(quad, oracle.moe_experts(x, w1, w2, wts, ids), dtype, "quad tile, experts only")
        _assert_close(whole, oracle.moe_experts(x, w1, w2, wts, ids), dtype, "quad tile, no tail split")
        # the layer with gating: top-2 of 8 experts, token rows gathered by sorted id, padding rows not fetched
        x2, logits, w1b, w2b = _inputs(1500, 1024, 1024, 8, 78, dtype)
        with fr.tunables(block=256):
            a = fused_moe(x2.cuda(), w1b.cuda(), w2b.cuda(), logits.cuda(), 2, True)
        with fr.tunables(block=256, no_quad=True):
            b = fused_moe(x2.cuda(), w1b.cuda(), w2b.cuda(), logits.cuda(), 2, True)
        torch.cuda.synchronize()
        assert torch.equal(a, b), "the two 256-row kernels differ (layer with gating)"
        _assert_close(a, oracle.fused_moe(x2, w1b, w2b, logits, 2, True), dtype, "quad tile, layer")
        # widths that are no multiples of 256: 18 and 22 K tiles, the down projection's last feature tile half wide;
        # three experts, one of them without a token
        x3, logits3, w1c, w2c = _inputs(900, 1152, 1408, 3, 79, dtype)
        logits3[:, 1] = -30.0
        with fr.tunables(block=256):
            c = fused_moe(x3.cuda(), w1c.cuda(), w2c.cuda(), logits3.cuda(), 2, True)
        with fr.tunables(block=256, no_quad=True):
            d = fused_moe(x3.cuda(), w1c.cuda(), w2c.cuda(), logits3.cuda(), 2, True)
        torch.cuda.synchronize()
        assert torch.equal(c, d), "the two 256-row kernels differ (odd widths)"
        _assert_close(c, oracle.fused_moe(x3, w1c, w2c, logits3, 2, True), dtype, "quad tile, odd widths")
    finally:
        fr.reset_tunables()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", ["heights", "many_experts", "odd_width", "plan_of_128", "plan_of_160"])
def test_tiles_as_tall_as_the_experts_runs(native, kernels_of, dtype, case):
    """The one-wavefront-per-SIMD kernel cuts an expert's run into tiles of 1 to 9 units of 32 rows, whatever the routing
    block.  heights: runs that end one slot before, at and behind every unit, of one to five tiles, and an expert without a
    pair; many_experts: 130 experts (more than a wavefront's lanes) with a
    few pairs each and two long runs; odd_width: the staged entry points at widths whose last feature tile starts early
    (F = 1088, H = 1152), with prepared weights, too; plan_of_128 / plan_of_160: layers whose plan routes for smaller blocks and leaves the heights to the
    kernel."""
    import fast_route_amd as fr
    from fast_route_amd import fused_experts, fused_moe
    from fast_route_amd.layers.fused_moe import plan
    _say(f"tile heights {case} {dtype}")
    if case.startswith("plan_of"):
        M, H, Fd, E, k = (1350, 4096, 2048, 8, 2) if case == "plan_of_128" else (2250, 4096, 2048, 8, 2)
        assert plan(M, H, Fd, E, k, dtype).block == int(case[-3:])
        x, logits, w1, w2 = _inputs(M, H, Fd, E, 83, dtype)
        args = [t.cuda() for t in (x, w1, w2, logits)]
        out, names = kernels_of(lambda: fused_moe(*args, k, True))
        assert sum("moe_gemm_quad_kernel" in n for n in names) == 2, names
        _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, case)
        return
    H, Fd = (1152, 1088) if case == "odd_width" else (1024, 1024)
    if case == "many_experts":
        counts = [1 + (e * 7) % 5 for e in range(130)]
        counts[3], counts[64], counts[129] = 700, 0, 290
    else:
        counts = [32 * u + d for u in range(1, 10) for d in (-1, 0, 1)] + [0, 320, 289, 575, 800, 1060, 1]
    ids = torch.from_numpy(np.repeat(np.arange(len(counts)), counts)).int()
    ids = ids[torch.from_numpy(np.random.default_rng(6).permutation(ids.numel()))].view(-1, 1)
    M, E = ids.shape[0], len(counts)
    x, _, w1, w2 = _inputs(M, H, Fd, E, 82, dtype)
    wts = torch.rand(M, 1) + 0.5
    args = [t.cuda() for t in (x, w1, w2, wts, ids)]

    def staged(x, w1, w2, wts, ids, flags=0):
        from fast_route_amd import _native as N
        from fast_route_amd.ops.fused_moe import moe_align_block_size
        s, e, npost = moe_align_block_size(ids, 256, E)
        act = torch.zeros(s.numel(), Fd, dtype=dtype, device="cuda")
        partial = torch.empty(M * H, dtype=torch.float32, device="cuda")
        out = torch.empty(M, H, dtype=dtype, device="cuda")
        lib, st, code = N.lib(), torch.cuda.current_stream().cuda_stream, N.dtype_code(dtype) | flags
        N.check(lib.fr_moe_gateup_silu(x.data_ptr(), w1.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(), M, H, Fd, E, 1, 256, code,
                                       act.data_ptr(), None, st))
        N.check(lib.fr_moe_down_combine(act.data_ptr(), w2.data_ptr(), wts.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(), M, H,
                                        Fd, E, 1, 256, 1, code, partial.data_ptr(), out.data_ptr(), None, st))
        return out

    experts = staged if case == "odd_width" else fused_experts
    try:
        with fr.tunables(block=256):
            out = experts(*args)
        with fr.tunables(block=256, no_quad=True):
            eight = experts(*args)
        if case == "odd_width":
            from fast_route_amd.layers.fused_moe import prepare_weights
            p1, p2, flags = prepare_weights(args[1], args[2], "both")
            assert torch.equal(staged(args[0], p1, p2, *args[3:], flags), out), "prepared weights"
        torch.cuda.synchronize()
    finally:
        fr.reset_tunables()
    _assert_close(out, oracle.moe_experts(x, w1, w2, wts, ids), dtype, case)
    # K below 4096 puts the eight-wavefront kernel on 32x32 MFMAs: the same products, another order of the sums inside one
    # MFMA, so up to an ulp of the operand type after the two roundings on the way
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert ((out.float() - eight.float()).abs() <= 2 * ulp * eight.float().abs().max()).all()


@pytest.mark.parametrize("M,H,Fd,E,k,planned,rows", [
    # many narrow experts: pairs per expert, w2 rows of other lengths and of a power of two, gate/up rows above 4 KB, wide experts
    (15, 2048, 640, 32, 4, 16, 16), (16, 2048, 640, 32, 4, 16, 32), (64, 2048, 640, 32, 4, 16, 32), (95, 2048, 640, 32, 4, 32, 32), (96, 2048, 640, 32, 4, 32, 64),
    (223, 2048, 640, 32, 4, 32, 64), (224, 2048, 640, 32, 4, 32, 128), (255, 2048, 640, 32, 4, 32, 128), (191, 2048, 512, 32, 4, 32, 32), (192, 2048, 512, 32, 4, 32, 64),
    (96, 2048, 1024, 32, 4, 32, 64), (191, 2048, 2048, 32, 4, 32, 32), (192, 2048, 2048, 32, 4, 32, 64), (16, 2048, 256, 32, 4, 16, 32), (230, 2048, 256, 32, 4, 32, 32),
    (32, 2176, 640, 32, 4, 16, 16), (16, 2048, 2176, 32, 4, 16, 16),
    # H of 640 to 1024: gate/up tiles with one block per expert, pairs per expert, K slices
    (36, 1024, 3584, 8, 2, 32, 64), (417, 1024, 3584, 8, 2, 128, 128), (416, 1024, 3584, 8, 2, 128, 64), (40, 1024, 4096, 8, 2, 32, 16), (41, 1024, 4096, 8, 2, 32, 32),
    (192, 1024, 4096, 8, 2, 128, 64), (193, 1024, 4096, 8, 2, 128, 128), (36, 1024, 2048, 8, 2, 32, 32), (125, 1024, 2048, 2, 2, 128, 64), (126, 1024, 2048, 2, 2, 128, 128),
    (72, 1024, 1536, 16, 2, 32, 64), (300, 1024, 1536, 16, 2, 128, 128), (180, 1024, 2048, 4, 2, 128, 64), (253, 1024, 2048, 8, 2, 128, 64), (361, 1024, 2048, 8, 2, 128, 128), (36, 896, 3584, 8, 2, 32, 32),
    (900, 4096, 1024, 16, 2, 128, 160)])
def test_layers_route_for_another_block_than_the_plan(native, kernels_of, M, H, Fd, E, k, planned, rows):
    """At the edges of the ranges where the layers take other tiles than the plan's block stands for: the plan stays, its workspace
    covers both, and results match the oracle."""
    from fast_route_amd import fused_experts, fused_moe
    from fast_route_amd.layers.fused_moe import plan, prepare_weights
    dtype = torch.bfloat16
    _say(f"layer's own block M={M} H={H} F={Fd} E={E}")
    assert plan(M, H, Fd, E, k, dtype).block == planned
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 3 + M, dtype, zipf=E >= 32)
    args = [x.cuda(), w1.cuda(), w2.cuda()]
    out, names = kernels_of(lambda: fused_moe(*args, logits.cuda(), k, True))
    tiles = {int(n) for x in names if "moe_gemm" in x for n in re.findall(r"Cfg(?:ILi|<)(\d+)", x)}
    assert tiles == {rows}, names
    w, ids = oracle.gating_topk(logits, k, True)
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, "layer")
    _assert_close(fused_experts(*args, w.cuda(), ids.cuda()), oracle.moe_experts(x, w1, w2, w, ids), dtype, "experts")
    t1, t2, flags = prepare_weights(*args[1:], which="both")
    assert torch.equal(fused_moe(args[0], t1, t2, logits.cuda(), k, True, weights_prepared=flags), out)


@pytest.mark.parametrize("M,E,k,launches", [(32, 64, 6, 1), (33, 64, 6, 2), (31, 33, 4, 1), (33, 33, 4, 2), (64, 32, 4, 1), (65, 32, 4, 2),
                                            (192, 16, 2, 1), (193, 16, 2, 2), (128, 16, 3, 1), (129, 16, 3, 2), (384, 8, 2, 1), (385, 8, 2, 2),
                                            (16, 128, 8, 1), (17, 128, 8, 2), (16, 200, 6, 1), (17, 200, 6, 2)])
def test_gating_and_sort_in_one_launch_or_two(native, kernels_of, M, E, k, launches):
    """Both sides of the rule that leaves small batches' gating and sort to one workgroup; the layer matches the oracle."""
    from fast_route_amd import fused_moe
    dtype = torch.bfloat16
    _say(f"routing launches M={M} E={E} k={k}")
    x, logits, w1, w2 = _inputs(M, 128, 128, E, 5 + M, dtype)
    out, names = kernels_of(lambda: fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, True))
    assert sum("route_align_small" in n for n in names) == (launches == 1) and sum("gating_topk" in n for n in names) == (launches == 2), names
    _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, "layer")


@pytest.mark.parametrize("M,H,Fd,E,k", [(68, 2048, 256, 32, 4), (900, 4096, 1024, 16, 2), (1031, 4096, 4096, 8, 2)])
def test_layer_in_the_scratch_of_the_plans_own_block(native, M, H, Fd, E, k):
    """A workspace that holds the plan's block and tail buffers of 256 rows only: the layer stays inside it and matches the oracle."""
    import fast_route_amd as fr
    from fast_route_amd import _native
    from fast_route_amd.layers.fused_moe import plan
    dtype = torch.bfloat16
    _say(f"smaller workspace M={M} H={H} F={Fd} E={E}")
    p = plan(M, H, Fd, E, k, dtype)
    try:
        with fr.tunables(block=p.block, split_k=p.split_k):
            own = plan(M, H, Fd, E, k, dtype)
    finally:
        fr.reset_tunables()
    least = own.workspace_bytes - (256 * 256 * 4 * (288 - 256) if own.tail_bytes else 0)
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 3 + M, dtype)
    xd, ld, w1d, w2d = x.cuda(), logits.cuda(), w1.cuda(), w2.cuda()
    guard = 4096
    for n in (least, p.workspace_bytes):
        buf = torch.full((n + 2 * guard,), 0x5A, dtype=torch.uint8, device="cuda")
        ws, out = buf[guard:], torch.empty_like(xd)
        assert ws.data_ptr() % 256 == 0
        _native.check(_native.lib().fr_fused_moe(xd.data_ptr(), w1d.data_ptr(), w2d.data_ptr(), ld.data_ptr(), _native.dtype_code(ld.dtype), M, H, Fd,
                                                 E, k, 1, _native.dtype_code(dtype), out.data_ptr(), ws.data_ptr(), n, _native.stream_ptr(xd.device)))
        torch.cuda.synchronize()
        assert (buf[:guard] == 0x5A).all() and (buf[guard + n:] == 0x5A).all()
        _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, True), dtype, f"{n} bytes")


@pytest.mark.parametrize("M,Fd", [(645, 3200), (860, 7552)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_tile_per_expert_where_the_plan_has_two(native, kernels_of, dtype, M, Fd):
    """Runs of five to seven units that the plan's 128 or 160 rows cut in two: both GEMMs multiply them as one tile each, alone on its
    weight tile (K loop from a place of its own; 25 and 59 feature tiles, the last round cut).  One expert has a run of 8 units and
    one of 9 (no loop of its own), one a single pair and one none."""
    from fast_route_amd import fused_experts
    from fast_route_amd.layers.fused_moe import plan
    H, E, k = 4096, 8, 2
    _say(f"one tile per expert M={M} F={Fd} {dtype}")
    n = M * k
    counts = np.array([1, 0, 250, 260, 0, 0, 0, 0])
    counts[4:] = (n - counts.sum()) // 4
    counts[4] += n - counts.sum()
    rng = np.random.default_rng(M)
    ids = torch.from_numpy(rng.permutation(np.repeat(np.arange(E), counts))).int().view(M, k)
    x, _, w1, w2 = _inputs(M, H, Fd, E, 11 + M, dtype)
    wts = torch.rand(M, k, generator=torch.Generator().manual_seed(M)) + 0.5
    args = [x.cuda(), w1.cuda(), w2.cuda(), wts.cuda(), ids.cuda()]
    assert plan(M, H, Fd, E, k, dtype).block in (128, 160)
    out, names = kernels_of(lambda: fused_experts(*args))
    assert sum("moe_gemm_quad_kernel" in x for x in names) == 2, names
    assert torch.equal(out, fused_experts(*args))
    _assert_close(out, oracle.moe_experts(x, w1, w2, wts, ids), dtype, "one tile per expert")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, "fp8"])
@pytest.mark.parametrize("counts,tall", [((162, 162, 161, 161, 161, 161, 161, 161), True), ((330, 165, 165, 165, 165, 100, 100, 100), True),
                                         ((330, 330, 165, 165, 100, 100, 50, 50), False), ((170, 170, 158, 158, 158, 158, 159, 159), True), ((170, 160, 160, 160, 160, 160, 160, 160), False),
                                         ((645, 400, 0, 200, 44, 1, 0, 0), False)])
def test_skewed_runs_keep_the_plans_tiles(native, dtype, counts, tall):
    """Where near-uniform loads would make every expert's run one tall tile, the experts' runs decide: tall tiles with one run of
    three blocks among eight experts, the plan's tiles (bit for bit those of no_quad) with two, with one run of two blocks and with a
    skewed load; without cut tiles as well."""
    import fast_route_amd as fr
    from fast_route_amd import _native as N, fused_experts, fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd.layers.fused_moe import plan
    M, H, Fd, E, k = 645, 4096, 3328, 8, 2
    _say(f"tiles by runs {counts} {dtype}")
    pairs = np.repeat(np.arange(E), counts).reshape(k, M).T  # an expert's pairs are consecutive: no token has one twice
    pairs = torch.from_numpy(np.random.default_rng(5).permutation(pairs)).int().contiguous()
    two_byte = torch.bfloat16 if dtype == "fp8" else dtype
    assert plan(M, H, Fd, E, k, two_byte, N.FR_FP8_E4M3 if dtype == "fp8" else None).block == 160
    g = torch.Generator(device="cuda").manual_seed(len(set(counts)))
    x = torch.randn(M, H, generator=g, device="cuda").to(two_byte)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).to(two_byte)
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).to(two_byte)
    if dtype == "fp8":
        logits = torch.full((M, E), -8.0)
        logits.scatter_(1, pairs.long(), 2.0)
        args = [x, *prepare_weights_fp8(w1, w2), logits.cuda()]
        run = lambda: fused_moe_fp8(*args, k, True)
        ref = oracle.fused_moe_fp8(x.cpu(), w1.cpu(), w2.cpu(), logits, k, True)[0]
    else:
        wts = torch.full((M, k), 0.5)
        args = [x, w1, w2, wts.cuda(), pairs.cuda()]
        run = lambda: fused_experts(*args)
        ref = oracle.moe_experts(x.cpu(), w1.cpu(), w2.cpu(), wts, pairs)
    out, again = run(), run()
    try:
        with fr.tunables(no_quad=True):
            tiles = run()
        with fr.tunables(no_tail_split=True):
            whole = run()
            with fr.tunables(no_tail_split=True, no_quad=True):
                whole_tiles = run()
    finally:
        fr.reset_tunables()
    assert torch.equal(out, again)
    assert torch.equal(out, tiles) != tall and torch.equal(whole, whole_tiles) != tall
    for o in (out, tiles, whole):
        if dtype == "fp8":
            o = o.float().cpu()
            assert (o - ref).norm() / ref.norm() <= 1e-2 and (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()
        else:
            _assert_close(o, ref, dtype, f"{counts}")


@pytest.mark.parametrize("Fd,counts,tall", [
    (7296, (232,) * 8, True), (7296, (265,) * 3 + (212,) * 4 + (213,), True), (7296, (265,) * 4 + (199,) * 4, False), (7296, (400, 232, 232, 232, 200, 200, 180, 180), True),
    (10240, (232,) * 8, False), (10240, (265,) + (227,) * 5 + (228,) * 2, True), (10240, (265,) * 4 + (199,) * 4, False)])
def test_runs_that_nearly_fill_two_blocks(native, Fd, counts, tall):
    """128-row blocks and a mean run of nearly two of them: tall tiles with up to three runs of three blocks among eight experts; with
    10240 features, where two blocks each are whole rounds of tiles and one tall tile each is not, with at least one."""
    import fast_route_amd as fr
    from fast_route_amd import fused_experts
    from fast_route_amd.layers.fused_moe import plan
    M, H, E, k = 928, 4096, 8, 2
    _say(f"runs of nearly two blocks {Fd} {counts}")
    assert plan(M, H, Fd, E, k, torch.bfloat16).block == 128
    pairs = np.repeat(np.arange(E), counts).reshape(k, M).T
    pairs = torch.from_numpy(np.random.default_rng(5).permutation(pairs)).int().contiguous()
    g = torch.Generator(device="cuda").manual_seed(Fd)
    normal = lambda std, *shape: torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=g)
    args = [normal(1.0, M, H), normal(0.02, E, 2 * Fd, H), normal(0.02, E, H, Fd), torch.full((M, k), 0.5, device="cuda"), pairs.cuda()]
    out, again = fused_experts(*args), fused_experts(*args)
    with fr.tunables(no_quad=True):
        tiles = fused_experts(*args)
    assert torch.equal(out, again) and torch.equal(out, tiles) != tall
    _assert_close(out, tiles.cpu(), torch.bfloat16, "tall tiles against the plan's")


@pytest.mark.parametrize("M,H,Fd,E,k,quad", [(1350, 4096, 2048, 8, 2, 2), (1430, 4096, 2048, 8, 2, 2), (2300, 2048, 2048, 8, 2, 2),
                                              (1200, 4096, 2048, 8, 2, 0), (2100, 2048, 2048, 8, 2, 0), (2850, 1024, 3584, 8, 2, 0),
                                              (350, 4096, 2048, 1, 1, 0), (1055, 2048, 5632, 4, 2, 0)])
def test_layers_and_staged_entry_points_take_the_same_kernels(native, kernels_of, M, H, Fd, E, k, quad):
    """Layers whose plan routes for 128 or 160 rows: the one-wavefront-per-SIMD kernel for both GEMMs where the rule says so -
    enough pairs per expert (at the first and behind the last count of every hidden size), enough tiles, one K slice -, the
    plan's tiles elsewhere and under no_quad; the stage-by-stage twin, on the staged entry points with the plan's block,
    takes the layer's kernels and has its result."""
    import fast_route_amd as fr
    from fast_route_amd.layers import profile_fused_route, stable_route
    from fast_route_amd.layers.fused_moe import plan
    _say(f"route of plans of 128 / 160 rows M={M} H={H} F={Fd} E={E}")
    assert plan(M, H, Fd, E, k, torch.bfloat16).block in (128, 160)
    g = torch.Generator(device="cuda").manual_seed(96)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    gate = (torch.randn(H, E, generator=g, device="cuda") / 64).bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).bfloat16()
    count = lambda names: sum("moe_gemm_quad_kernel" in n for n in names)
    out, names = kernels_of(lambda: stable_route.fused_moe(x, gate, w1, w2, k, True))
    assert count(names) == quad, names
    with tempfile.TemporaryDirectory() as d:
        twin, names = kernels_of(lambda: profile_fused_route.fused_moe(x, gate, w1, w2, k, True, save_dir=d))
    assert count(names) == quad, names
    assert torch.equal(out, twin)
    with fr.tunables(no_quad=True):
        tiles, names = kernels_of(lambda: stable_route.fused_moe(x, gate, w1, w2, k, True))
    assert count(names) == 0, names
    _assert_close(out, tiles.cpu(), torch.bfloat16, "one-wavefront-per-SIMD kernel against the plan's tiles")


@pytest.mark.parametrize("M,H,Fd,E,k", [(900, 4096, 1024, 16, 2), (96, 2048, 640, 32, 4), (32, 2048, 1408, 64, 6), (240, 2048, 640, 32, 4), (130, 1024, 3584, 8, 2), (40, 1024, 4096, 8, 2),
                                        (1031, 4096, 4096, 8, 2), (1056, 4096, 2048, 8, 2), (645, 4096, 4096, 8, 2), (2050, 4096, 2048, 8, 2), (3, 4096, 1024, 8, 2)])
def test_stage_by_stage_twin_has_the_layers_result(native, kernels_of, M, H, Fd, E, k):
    """The twin on the staged entry points runs the layer's kernels and has its result bit for bit: where the layer routes for another block
    than the plan's, and where tiles are cut into as many slices as the layer's tail scratch has buffers for."""
    from fast_route_amd.layers import profile_fused_route, stable_route
    _say(f"twin M={M} H={H} F={Fd} E={E}")
    g = torch.Generator(device="cuda").manual_seed(96)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    gate = (torch.randn(H, E, generator=g, device="cuda") / 64).bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).bfloat16()
    gemms = lambda names: [n for n in names if "moe_gemm" in n or "rows_kernel" in n]
    out, names = kernels_of(lambda: stable_route.fused_moe(x, gate, w1, w2, k, True))
    with tempfile.TemporaryDirectory() as d:
        twin, twins = kernels_of(lambda: profile_fused_route.fused_moe(x, gate, w1, w2, k, True, save_dir=d))
    assert gemms(names) == gemms(twins)
    assert torch.equal(out, twin)


def test_more_than_64_tiles_per_workgroup(native, kernels_of):
    """The one-wavefront-per-SIMD kernel works a workgroup's tiles out 64 at a time: 131 tiles of up to 288 rows x 128 feature
    tiles on 256 workgroups are 65 or 66 each.  Operands are small integers, whose sums are exact in any order: equal to the
    eight-wavefront kernel bit for bit."""
    import fast_route_amd as fr
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    _say("more than 64 tiles per workgroup")
    M, N_, K = 37500, 32768, 1024
    g = torch.Generator(device="cuda").manual_seed(99)
    a = torch.randint(-1, 2, (M, K), generator=g, device="cuda").bfloat16()
    b = torch.randint(-1, 2, (1, N_, K), generator=g, device="cuda").bfloat16()
    ids = torch.zeros(M, 1, dtype=torch.int32, device="cuda")
    s, e, npost = moe_align_block_size(ids, 256, 1)
    res = []
    for no_quad in (False, True):
        c = torch.zeros(M, 1, N_, dtype=torch.bfloat16, device="cuda")
        with fr.tunables(no_quad=no_quad):
            _, names = kernels_of(lambda: invoke_fused_moe_kernel(a, b, c, None, ids, s, e, npost, False, 1, {"BLOCK_SIZE_M": 256}))
        assert any("moe_gemm_quad_kernel" in n for n in names) != no_quad, names
        res.append(c)
    assert torch.equal(res[0], res[1])
    rows = torch.tensor([0, 287, 288, 20000, M - 1], device="cuda")
    assert torch.equal(res[0][rows, 0], (a[rows].float() @ b[0].float().t()).bfloat16())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,E,Fd,cut", [(256, 8, 4096, ""), (256, 7, 4096, "down"), (288, 17, 2048, "gate/up, down"),
                                           (257, 17, 2048, "gate/up, down"), (545, 9, 2048, "gate/up, down")])
def test_cut_tiles_equal_whole_ones(native, rows, E, Fd, cut, dtype):
    """The last round's tiles cut along K by the one-wavefront-per-SIMD kernel: tiles of 256 rows, in the down projection of 8
    experts with every slice buffer of the layer's scratch in use (16 tiles per XCD in 2 slices; the staged entry points keep
    their list of cut tiles in the scratch and have one buffer less: not cut there), and tiles of 9 units (buffers of 288
    rows).  Operands are small integers times powers of two, whose sums are exact in any order: a cut tile equals the whole
    one bit for bit (fp16: up to the one rounding more of the fix-up launch)."""
    import fast_route_amd as fr
    from fast_route_amd import _native as N, fused_experts
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    H, M = 4096, rows * E
    _say(f"cut tiles rows={rows} E={E} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(94)
    ints = lambda hi, *shape: torch.randint(-hi, hi + 1, shape, generator=g, device="cuda").to(dtype)
    x, act_in, w1, w2 = ints(1, M, H), ints(2, M + E * 255, Fd), ints(1, E, 2 * Fd, H) / 64, ints(1, E, H, Fd) / 64
    x[:, 0] = 1
    w1[:, :Fd] = 0
    w1[:, :Fd, 0] = 64  # silu(64) is 64: the activated rows are sums times a power of two
    ids = (torch.randperm(M, generator=g, device="cuda") % E).int().view(M, 1)
    wts = torch.rand(M, 1, generator=g, device="cuda") + 0.5
    lib, st, code = N.lib(), torch.cuda.current_stream().cuda_stream, N.dtype_code(dtype)
    s, e, npost = moe_align_block_size(ids, 256, E)
    tail = torch.full((256 * 256 * 256,), float("nan"), dtype=torch.float32, device="cuda")
    pairs = (s < M).nonzero().view(-1)

    def gate_up(scratch):
        act = torch.zeros(s.numel(), Fd, dtype=dtype, device="cuda")
        N.check(lib.fr_moe_gateup_silu(x.data_ptr(), w1.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(), M, H, Fd, E, 1,
                                       256, code, act.data_ptr(), scratch, st))
        return act

    def down(act, scratch):
        partial = torch.empty(M * H, dtype=torch.float32, device="cuda")
        out = torch.empty(M, H, dtype=dtype, device="cuda")
        N.check(lib.fr_moe_down_combine(act.data_ptr(), w2.data_ptr(), wts.data_ptr(), s.data_ptr(), e.data_ptr(), npost.data_ptr(),
                                        M, H, Fd, E, 1, 256, 1, code, partial.data_ptr(), out.data_ptr(), scratch, st))
        return out

    def equal(a, b, what):
        if dtype == torch.bfloat16:
            assert torch.equal(a, b), what
        else:  # an ulp: 2^-10 of the value
            assert ((a.float() - b.float()).abs() <= 2.0 ** -10 * b.float().abs()).all(), what

    for name, run in (("gate/up", lambda t: gate_up(t)[pairs]), ("down", lambda t: down(act_in, t))):
        tail.fill_(float("nan"))
        out = run(tail.data_ptr())
        torch.cuda.synchronize()
        buffers = tail[: 8 * 28 * 288 * 256]  # without the list of cut tiles
        assert bool((~torch.isnan(buffers)).any()) == (name in cut), name
        assert torch.isfinite(out.float()).all()
        equal(out, run(None), name)
    with fr.tunables(block=256, split_k=1):
        layer = fused_experts(x, w1, w2, wts, ids)
    with fr.tunables(block=256, split_k=1, no_tail_split=True):
        equal(layer, fused_experts(x, w1, w2, wts, ids), "layer")
    equal(layer, down(gate_up(tail.data_ptr()), tail.data_ptr()), "layer and staged entry points")


@pytest.mark.parametrize("M,H,Fd,E,k", [(1055, 2048, 5632, 4, 2), (2150, 1024, 3584, 8, 2), (328, 4096, 4096, 2, 2)])
def test_a_plan_of_several_k_slices_keeps_their_fp32_rows(native, M, H, Fd, E, k):
    """Runs that would suit the one-wavefront-per-SIMD kernel (it writes a pair's row once, in the operands' type) under a
    plan of several K slices: the slices are summed from fp32 rows, as without that kernel, bit for bit."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    from fast_route_amd.layers.fused_moe import plan
    _say(f"K slices in fp32 M={M} H={H} F={Fd} E={E}")
    p = plan(M, H, Fd, E, k, torch.bfloat16)
    assert p.split_k > 1 and p.block in (128, 160)
    g = torch.Generator(device="cuda").manual_seed(90)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).bfloat16()
    logits = torch.randn(M, E, generator=g, device="cuda")
    out = fused_moe(x, w1, w2, logits, k, True)
    with fr.tunables(no_quad=True):
        q = plan(M, H, Fd, E, k, torch.bfloat16)
        assert (q.block, q.split_k) == (p.block, p.split_k)
        assert torch.equal(out, fused_moe(x, w1, w2, logits, k, True))


@pytest.mark.parametrize("E,k,H", [(8, 2, 4096), (64, 6, 4096), (100, 3, 4096), (256, 8, 4096), (4, 4, 4096), (16, 1, 4096),
                                   (64, 6, 2048), (8, 2, 3072), (16, 4, 2560)])
@pytest.mark.parametrize("ldtype", [torch.float32, torch.bfloat16])
def test_decode_layer_routes_inside_the_gate_up_launch(native, E, k, H, ldtype):
    """Up to 4 tokens with H >= 2048: fused_moe's gate/up launch gates the tokens and sorts the pairs itself.
    Its result must equal, bit for bit, the experts-only entry point fed with the gating kernel's weights and ids
    (the same gating core, the same routing order), and match the oracle; exact ties in the logits included."""
    from fast_route_amd import fused_moe, fused_experts
    from fast_route_amd.ops.stable_route import topk_softmax
    Fd, dtype = 256, torch.bfloat16
    _, _, w1, w2 = _inputs(1, H, Fd, E, 9, dtype)
    w1d, w2d = w1.cuda(), w2.cuda()
    for M in (1, 2, 3, 4):
        if M * k > 32:
            continue
        for renorm in (True, False):
            _say(f"routed decode E={E} k={k} H={H} {ldtype} M={M} renorm={renorm}")
            g = torch.Generator().manual_seed(E * 100 + k * 10 + M)
            x = torch.randn(M, H, generator=g).to(dtype)
            logits = torch.randn(M, E, generator=g).to(ldtype)
            if E >= 4:
                logits[0, : min(E, 5)] = logits[0, 0]  # a run of equal logits: lower index first
            out = fused_moe(x.cuda(), w1d, w2d, logits.cuda(), k, renorm)
            torch.cuda.synchronize()
            w = torch.empty((M, k), dtype=torch.float32, device="cuda")
            ids = torch.empty((M, k), dtype=torch.int32, device="cuda")
            topk_softmax(w, ids, None, logits.cuda(), renormalize=renorm)
            ow, oid = oracle.gating_topk(logits, k, renorm)
            assert torch.equal(ids.cpu(), oid)
            same = fused_experts(x.cuda(), w1d, w2d, w, ids)
            assert torch.equal(out, same), "routing inside the gate/up launch differs from the routing kernels"
            _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, renorm), dtype, f"routed decode M={M}")


def test_random_shapes_against_oracle(native):
    """Forty seeded random layer shapes (token count, widths, expert count, top-k, dtype, renormalisation)
    against the oracle: every plan boundary gets neighbours on both sides sooner or later."""
    from fast_route_amd import fused_moe
    rng = np.random.default_rng(20240607)
    for case in range(40):
        E = int(rng.choice([1, 2, 3, 4, 8, 16, 60, 64]))
        k = int(rng.integers(1, min(E, 8) + 1))
        H = int(rng.choice([128, 256, 384, 512, 1024, 2048, 3072, 4096]))
        Fd = int(rng.choice([128, 256, 384, 640]))
        M = int(rng.choice([1, 2, 3, 4, 5, 7, 17, 33, 100, 257, 600]) if rng.random() < 0.7 else rng.integers(1, 700))
        dtype = torch.bfloat16 if rng.random() < 0.7 else torch.float16
        renorm = bool(rng.random() < 0.7)
        _say(f"random case {case}: M={M} H={H} F={Fd} E={E} k={k} {dtype} renorm={renorm}")
        x, logits, w1, w2 = _inputs(M, H, Fd, E, 1000 + case, dtype, zipf=bool(rng.random() < 0.3))
        out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), k, renorm)
        torch.cuda.synchronize()
        _assert_close(out, oracle.fused_moe(x, w1, w2, logits, k, renorm), dtype, f"random case {case}")


@pytest.mark.parametrize("M,E,k,H,Fd", [(2, 8, 2, 512, 4096), (3, 8, 2, 512, 1024), (300, 8, 2, 512, 1024), (700, 8, 2, 512, 1024),
                                        (200, 64, 6, 512, 384)])
def test_out_of_range_expert_ids_are_dropped_pairs(native, M, E, k, H, Fd):
    """Expert ids outside [0, E) (masked pairs of an expert-parallel caller) get no slot in the routing arrays
    and contribute nothing: the oracle's per-expert masks never match them either (perf_test_moe.py:22-27).
    Covers the decode kernels, the combine in the GEMM epilogue (top-2) and the combine kernel (top-6);
    with every pair masked the output is exactly zero."""
    from fast_route_amd import fused_experts
    dtype = torch.bfloat16
    _say(f"masked ids M={M} E={E} k={k}")
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 31, dtype)
    tw, ti = oracle.gating_topk(logits, k, True)
    g = torch.Generator().manual_seed(M)
    drop = torch.rand(M, k, generator=g) < 0.3
    ti = ti.clone()
    ti[drop] = torch.where(torch.rand(int(drop.sum()), generator=g) < 0.5, -1, E + 3).int()
    xd, w1d, w2d = x.cuda(), w1.cuda(), w2.cuda()
    out = fused_experts(xd, w1d, w2d, tw.cuda(), ti.cuda())
    torch.cuda.synchronize()
    _assert_close(out, oracle.moe_experts(x, w1, w2, tw, ti), dtype, f"masked ids M={M}")
    none = torch.full_like(ti, -1)
    out0 = fused_experts(xd, w1d, w2d, tw.cuda(), none.cuda())
    torch.cuda.synchronize()
    assert torch.count_nonzero(out0) == 0, "all pairs masked: output must be zero"


@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8])
def test_combine_over_every_slot_count(native, k, split):
    """The combine kernel takes the rows of two, three or four slots at a time: every remainder, over one and two K
    slices, with dropped pairs whose rows are never written (the scratch is filled with NaN beforehand)."""
    from fast_route_amd import _native as N
    from fast_route_amd import fused_experts
    from fast_route_amd.layers.fused_moe import workspace
    M, E, H, Fd = 70, 12, 512, 2048  # 8 K tiles of the 16-row block's 128 elements per slice: k = 1 is really cut in two
    _say(f"combine k={k} split={split}")
    x, logits, w1, w2 = _inputs(M, H, Fd, E, 53, torch.bfloat16)
    tw, ti = oracle.gating_topk(logits, k, True)
    ti = ti.clone()
    ti[torch.rand(M, k, generator=torch.Generator().manual_seed(k)) < 0.25] = E
    t = N.FrMoeTunables()
    t.split_k = split
    N.check(N.lib().fr_moe_set_tunables(t))
    try:
        ws = workspace(M, H, Fd, E, k, torch.bfloat16, "cuda").fill_(0xFF)
        out = fused_experts(x.cuda(), w1.cuda(), w2.cuda(), tw.cuda(), ti.cuda(), workspace_buf=ws)
        torch.cuda.synchronize()
    finally:
        N.check(N.lib().fr_moe_set_tunables(None))
    _assert_close(out, oracle.moe_experts(x, w1, w2, tw, ti), torch.bfloat16, f"combine k={k} split={split}")


@pytest.mark.parametrize("split,Fd", [(1, 4096), (2, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sixteen_row_down_projection_over_several_rounds(native, dtype, split, Fd):
    """The 16-row down projection with 8 KB of K per slice is persistent: 42 blocks x 16 feature tiles are more than its
    512 workgroups (two K slices: 256 each), so workgroups hand their ring over to a second and third tile - between full
    blocks, blocks of one pair and the two blocks of an expert with 17 pairs."""
    from fast_route_amd import _native as N
    from fast_route_amd import fused_experts
    E, H = 40, 1024
    _say(f"16-row down rounds {dtype} split={split}")
    g = torch.Generator().manual_seed(91)
    counts = [(16, 1, 9, 17)[e % 4] if e < 8 else 1 + (e * 7) % 16 for e in range(E)]
    ti = torch.repeat_interleave(torch.arange(E, dtype=torch.int32), torch.tensor(counts))
    M = ti.numel()
    ti = ti[torch.randperm(M, generator=g)].view(M, 1).contiguous()
    gd = torch.Generator(device="cuda").manual_seed(92)
    w1 = torch.empty(E, 2 * Fd, H, dtype=dtype, device="cuda").normal_(0, 0.02, generator=gd)
    w2 = torch.empty(E, H, Fd, dtype=dtype, device="cuda").normal_(0, 0.02, generator=gd)
    x = torch.randn(M, H, generator=g).to(dtype).cuda()
    tw = torch.rand(M, 1, generator=g).cuda()
    t = N.FrMoeTunables()
    t.block, t.split_k = 16, split
    N.check(N.lib().fr_moe_set_tunables(t))
    try:
        out = fused_experts(x, w1, w2, tw, ti.cuda())
        torch.cuda.synchronize()
    finally:
        N.check(N.lib().fr_moe_set_tunables(None))
    ref = torch.empty(M, H)
    for e in range(E):
        rows = (ti[:, 0] == e).nonzero()[:, 0]
        h = x[rows.cuda()].float() @ w1[e].float().t()
        act = (torch.nn.functional.silu(h[:, :Fd]) * h[:, Fd:]).to(dtype).float()
        ref[rows] = ((act @ w2[e].float().t()) * tw[rows.cuda()]).cpu()
    _assert_close(out, ref, dtype, f"16-row down rounds split={split}")


@pytest.mark.parametrize("E", [3, 64, 256, 257, 300])
def test_persistent_tiles_with_experts_missing(native, E):
    """The walk table of the persistent tiles where most experts have no block (runs of equal entries at the front, in
    between and at the end), below and above the expert count up to which it is built in one pass."""
    from fast_route_amd.ops.fused_moe import invoke_fused_moe_kernel, moe_align_block_size
    n, N_, K, block = 700, 256, 512, 160  # 160 rows: persistent at op level too, from 5 K tiles on
    _say(f"experts missing E={E}")
    g = torch.Generator().manual_seed(E)
    used = torch.tensor(sorted({1, E // 3, E // 2, E - 2}))
    ids = used[torch.randint(0, len(used), (n, 1), generator=g)].int()
    a = (torch.randn(n, K, generator=g) / 8).bfloat16()
    b = (torch.randn(E, N_, K, generator=g) / 8).bfloat16()
    s, e, npost = moe_align_block_size(ids.cuda(), block, E)
    c = torch.zeros(n, 1, N_, dtype=torch.bfloat16, device="cuda")
    invoke_fused_moe_kernel(a.cuda(), b.cuda(), c, None, ids.cuda(), s, e, npost, False, 1, {"BLOCK_SIZE_M": block})
    torch.cuda.synchronize()
    ref = torch.stack([b[int(ids[p])].float() @ a[p].float() for p in range(n)])
    _assert_close(c.view(n, N_), ref, torch.bfloat16, f"experts missing E={E}")


@pytest.mark.parametrize("E", [8, 100, 256])
@pytest.mark.parametrize("M", [3, 40])
def test_nan_logit_rows_do_not_reach_the_weights(native, E, M):
    """A token whose router logits are all NaN has no valid expert (with more than 64 experts the gating core
    leaves an id outside [0, E) behind): its pairs are dropped by the routing - also by the routing done inside
    the decode gate/up launch - instead of indexing the weights, and the other tokens are unaffected."""
    from fast_route_amd import fused_moe
    dtype = torch.bfloat16
    _say(f"NaN logits E={E} M={M}")
    x, logits, w1, w2 = _inputs(M, 2048, 256, E, 13, dtype)
    logits = logits.clone()
    logits[1, :] = float("nan")
    out = fused_moe(x.cuda(), w1.cuda(), w2.cuda(), logits.cuda(), 2, True)
    torch.cuda.synchronize()
    keep = [m for m in range(M) if m != 1]
    ref = oracle.fused_moe(x[keep], w1, w2, logits[keep], 2, True)
    _assert_close(out[keep], ref, dtype, f"NaN logits E={E}")
    if E > 64:
        assert torch.count_nonzero(out[1]) == 0


@pytest.mark.parametrize("M", [40, 300, 3000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_top2_combine_in_the_epilogue_is_deterministic(native, M, dtype):
    """The epilogue_combine knob: top-2 layers add the two weighted rows of a token into a zero-filled output
    with packed atomics.  The result may not depend on which pair arrives first: same bits on every run, also
    in place, and the same bits as the combine kernel forms from the same two rounded rows."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe
    _say(f"top-2 epilogue combine M={M} {dtype}")
    x, logits, w1, w2 = _inputs(M, 512, 1024, 8, 17, dtype)
    xd, w1d, w2d, ld = x.cuda(), w1.cuda(), w2.cuda(), logits.cuda()
    with fr.tunables(split_k=1):
        by_kernel = fused_moe(xd, w1d, w2d, ld, 2, True)
    with fr.tunables(split_k=1, epilogue_combine=True):
        first = fused_moe(xd, w1d, w2d, ld, 2, True)
        for _ in range(4):
            assert torch.equal(fused_moe(xd, w1d, w2d, ld, 2, True), first)
        xin = xd.clone()
        assert torch.equal(fused_moe(xin, w1d, w2d, ld, 2, True, inplace=True), first)
    torch.cuda.synchronize()
    _assert_close(first, oracle.fused_moe(x, w1, w2, logits, 2, True), dtype, f"top-2 M={M}")
    assert torch.equal(first, by_kernel), "epilogue combine and combine kernel round differently"


_FIRST_CALL_CAPTURE = r'''
import sys
sys.path.insert(0, sys.argv[1])
import torch
import fast_route_amd as fr
from fast_route_amd import _native as N
from fast_route_amd.layers.fused_moe import plan

dtype, lib = torch.bfloat16, N.lib()
fr.prepare(dtype)                      # every kernel set up, the no-alloc scratch resolved: nothing left to do lazily
gen = torch.Generator().manual_seed(9)
cases = []
for M, H, Fd, E, k in ((2, 4096, 512, 4, 2), (16, 1024, 2048, 4, 2), (1536, 1024, 2048, 4, 2)):
    x = torch.randn(M, H, generator=gen).to(dtype).cuda()
    logits = torch.randn(M, E, generator=gen).cuda()
    w1 = (torch.randn(E, 2 * Fd, H, generator=gen) * 0.02).to(dtype).cuda()
    w2 = (torch.randn(E, H, Fd, generator=gen) * 0.02).to(dtype).cuda()
    p = plan(M, H, Fd, E, k, dtype)
    ws = torch.empty(max(p.workspace_bytes, 256), dtype=torch.uint8, device="cuda")
    out, out_na = torch.zeros(M, H, dtype=dtype, device="cuda"), torch.zeros(M, H, dtype=dtype, device="cuda")
    na = p.workspace_bytes <= (64 << 20)

    def call(stream, x=x, w1=w1, w2=w2, logits=logits, M=M, H=H, Fd=Fd, E=E, k=k, out=out, out_na=out_na, ws=ws, na=na):
        N.check(lib.fr_fused_moe(x.data_ptr(), w1.data_ptr(), w2.data_ptr(), logits.data_ptr(), N.FR_F32, M, H, Fd, E, k, 1,
                                 N.FR_BF16, out.data_ptr(), ws.data_ptr(), ws.numel(), stream))
        if na:
            N.check(lib.fr_fused_moe_noalloc(x.data_ptr(), w1.data_ptr(), w2.data_ptr(), logits.data_ptr(), N.FR_F32, M, H, Fd,
                                             E, k, 1, N.FR_BF16, out_na.data_ptr(), stream))
    cases.append((M, call, out, out_na, na))
torch.cuda.synchronize()
graphs = []
for M, call, out, out_na, na in cases:  # the captured calls are this process's first launches of these kernels
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call(torch.cuda.current_stream().cuda_stream)
    graphs.append(g)
for (M, call, out, out_na, na), g in zip(cases, graphs):
    for rep in range(2):
        out.zero_(); out_na.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got, got_na = out.clone(), out_na.clone()
        out.zero_(); out_na.zero_()
        call(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.count_nonzero(got) > 0
        assert torch.equal(got, out), "M=%d replay %d: captured first call differs from the eager call" % (M, rep)
        if na:
            assert torch.equal(got_na, out_na) and torch.equal(got_na, got), "M=%d: no-alloc entry under capture" % M
print("FIRST-CALL-CAPTURE-OK")
'''


def test_first_call_under_graph_capture_after_prepare(native):
    """What fr_moe_prepare exists for: in a fresh process, after fr_moe_prepare and nothing else, the whole layer -
    through fr_fused_moe and through fr_fused_moe_noalloc - is captured as the process's FIRST launch of its
    kernels (weight-row decode kernels, decode tiles with the fused route+align launch, persistent tiles with
    their last-round split) and replays to the bits of the eager calls made afterwards."""
    import os
    import subprocess
    _say("first call captured after fr_moe_prepare (fresh process)")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, "-c", _FIRST_CALL_CAPTURE, root], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=110)
    assert proc.returncode == 0 and "FIRST-CALL-CAPTURE-OK" in proc.stdout, proc.stdout[-3000:]
