"""GPU parity of the fp8 (e4m3fn) path.  The reference has no fp8 code, so the
oracle here is this build's own definition (dequantise -> fp32), see oracle/moe_oracle.py."""
import sys

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _say(msg):
    print("[case] " + msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_quantisation_bit_exact(native, dtype):
    from fast_route_amd import quantize_rows_e4m3
    # rows of up to 16384 elements are held in registers by a workgroup (2, 4 or 8 chunks per thread, the last
    # one partly filled); longer rows take the two-pass kernel
    for rows, K, std in ((1, 16, 1.0), (37, 1024, 1.0), (130, 4096, 0.02), (16, 14336, 3.0), (9, 5008, 1.0),
                         (3, 9008, 0.5), (4, 16384, 1.0), (5, 16400, 1.0)):
        _say(f"quant rows={rows} K={K} std={std} {dtype}")
        g = torch.Generator().manual_seed(rows * 7 + K)
        x = (torch.randn(rows, K, generator=g) * std).to(dtype)
        if rows > 2:
            x[1].zero_()                      # all-zero row -> scale 1, codes 0
            x[2, 5] = 448.0 if dtype == torch.bfloat16 else 400.0
        q, s = quantize_rows_e4m3(x.cuda())
        torch.cuda.synchronize()
        rq, rs = oracle.quant_e4m3_rows(x)
        assert np.array_equal(s.cpu().numpy(), rs), "scales differ"
        got, ref = q.cpu().numpy(), rq
        zero = (ref & 0x7F) == 0              # the sign of a zero code is not significant
        assert np.array_equal(got[~zero], ref[~zero]) and ((got[zero] & 0x7F) == 0).all(), "codes differ"


@pytest.mark.parametrize("M", [16, 64, 200, 700, 2048])
def test_fp8_layer_vs_oracle(native, M):
    """fp8 workload shape family (E8 top2) at reduced width; every tile plan is hit.
    Tolerance: the GPU and the oracle quantise the same bf16 activations, so they
    differ only by fp32 summation order, occasional 1-ulp flips of the bf16
    intermediate (and hence a few fp8 codes): ||out-ref||_F <= 1e-2 ||ref||_F and
    max|out-ref| <= 2**-5 max|ref|."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say(f"fp8 layer M={M}")
    H, Fd, E, k = 512, 1024, 8, 2
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=77)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
    out = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
    torch.cuda.synchronize()
    ref, parts = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    # the prepared weights are bit-identical to the oracle's
    assert np.array_equal(w1s.cpu().numpy(), parts["w1_scale"]) and np.array_equal(w2s.cpu().numpy(), parts["w2_scale"])
    z = (parts["w1_codes"] & 0x7F) == 0
    assert np.array_equal(w1q.cpu().numpy()[~z], parts["w1_codes"][~z])
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    rel = (o - ref).norm() / ref.norm()
    err = (o - ref).abs().max()
    assert rel <= 1e-2, f"rel F error {rel:.3e}"
    assert err <= 2.0 ** -5 * ref.abs().max(), f"max abs err {err:.3e}"
    # and it stays close to the unquantised fp32 layer (quantisation noise only)
    full = oracle.fused_moe(x, w1, w2, logits, k, True)
    assert (o - full).norm() / full.norm() < 0.08


@pytest.mark.parametrize("M", [1, 16, 200, 700, 2048])
def test_fp8_layer_does_not_use_padding_rows(native, M):
    """Padding slots' activated rows are not quantised: whatever the scratch held in their place (NaN codes and scales
    here, zeros there), the output is the same bit for bit."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd import _native as N
    from fast_route_amd.layers.fused_moe import plan
    _say(f"fp8 padding rows M={M}")
    H, Fd, E, k = 512, 1024, 8, 2
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=78)
    w = prepare_weights_fp8(w1.bfloat16().cuda(), w2.bfloat16().cuda())
    ws = torch.empty(plan(M, H, Fd, E, k, None, code=N.FR_FP8_E4M3).workspace_bytes, dtype=torch.uint8, device="cuda")
    outs = []
    for fill in (0xFF, 0):
        out = fused_moe_fp8(x.bfloat16().cuda(), *w, logits.cuda(), k, True, workspace_buf=ws.fill_(fill))
        torch.cuda.synchronize()
        outs.append(out.clone())
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("split,Fd", [(1, 8192), (2, 16384)])
def test_fp8_sixteen_row_down_projection_over_several_rounds(native, split, Fd):
    """Persistent 16-row tiles in fp8 (8 KB of K per slice of the down projection) with more tiles than workgroups: the ring
    is handed over between full blocks, blocks of one pair and the two blocks of an expert with 17 pairs.  Tolerance as for
    the layer against the oracle: the reference quantises the same activations, in fp32 on dequantised operands."""
    from fast_route_amd import _native as N
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8, quantize_rows_e4m3
    E, H = 40, 1024
    _say(f"fp8 16-row down rounds split={split}")
    g = torch.Generator().manual_seed(93)
    counts = [(16, 1, 9, 17)[e % 4] if e < 8 else 1 + (e * 7) % 16 for e in range(E)]
    ti = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    M = ti.numel()
    ti = ti[torch.randperm(M, generator=g)]
    logits = torch.randn(M, E, generator=g)
    logits[torch.arange(M), ti] += 20.0
    gd = torch.Generator(device="cuda").manual_seed(94)
    w = prepare_weights_fp8(torch.empty(E, 2 * Fd, H, dtype=torch.bfloat16, device="cuda").normal_(0, 0.02, generator=gd),
                            torch.empty(E, H, Fd, dtype=torch.bfloat16, device="cuda").normal_(0, 0.02, generator=gd))
    x = torch.randn(M, H, generator=g).bfloat16().cuda()
    t = N.FrMoeTunables()
    t.block, t.split_k = 16, split
    N.check(N.lib().fr_moe_set_tunables(t))
    try:
        out = fused_moe_fp8(x, *w, logits.cuda(), 1, True)
        torch.cuda.synchronize()
    finally:
        N.check(N.lib().fr_moe_set_tunables(None))

    def wide(codes, scale):
        return codes.view(torch.float8_e4m3fn).float() * scale[:, None]

    ref = torch.empty(M, H)
    xq = wide(*quantize_rows_e4m3(x))
    for e in range(E):
        rows = (ti == e).nonzero()[:, 0]
        h = xq[rows.cuda()] @ wide(w[0][e], w[1][e]).t()
        act = (torch.nn.functional.silu(h[:, :Fd]) * h[:, Fd:]).bfloat16()
        ref[rows] = (wide(*quantize_rows_e4m3(act)) @ wide(w[2][e], w[3][e]).t()).cpu()
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() <= 1e-2 * ref.norm() and (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_layer_with_64_row_blocks(native):
    """H = 4096 with 40 pairs per expert: the plan takes 64-row routing blocks for fp8 too."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd.layers.fused_moe import plan
    _say("fp8 layer with 64-row blocks")
    M, H, Fd, E, k = 160, 4096, 1024, 8, 2
    from fast_route_amd import _native as N
    assert plan(M, H, Fd, E, k, None, code=N.FR_FP8_E4M3).block == 64
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=64)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
    out = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
    torch.cuda.synchronize()
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_mixtral_shape_sampled(native):
    """Full fp8 workload shape (H4096 F14336 E8 top2), M in {16, 128, 256, 512, 1024, 4096} (512 and 1024: 160-row blocks): sampled tokens vs the
    oracle.  At M=4096 the down projection runs the persistent form with its last round of tiles
    split along K."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    H, Fd, E, k = 4096, 14336, 8, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).bfloat16()
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1, w2)
    w1c, w2c = w1.cpu(), w2.cpu()
    wq = oracle.quantize_weights_fp8(w1c, w2c)  # once: 1.4e9 weights through the CPU encoder
    for M in (16, 128, 256, 512, 1024, 4096):
        _say(f"fp8 mixtral M={M}")
        x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
        logits = torch.randn(M, E, generator=g, device="cuda")
        out = fused_moe_fp8(x, w1q, w1s, w2q, w2s, logits, k, True)
        torch.cuda.synchronize()
        sample = torch.arange(0, M, max(1, M // 12))[:12]
        ref, _ = oracle.fused_moe_fp8(x[sample].cpu(), w1c, w2c, logits[sample].cpu(), k, True, weights_q=wq)
        o = out[sample].float().cpu()
        assert (o - ref).norm() / ref.norm() <= 1e-2
        # same quantised operands on both sides: what is left is accumulation order and the bf16 rounding of
        # the activated row (which can flip an e4m3 code of its re-quantisation) and of the output: the bound of the other fp8 tests
        assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max(), f"M={M}: max abs err {(o - ref).abs().max():.3e} of {ref.abs().max():.3e}"
        out2 = fused_moe_fp8(x, w1q, w1s, w2q, w2s, logits, k, True)
        assert torch.equal(out, out2)


def test_fp8_down_projection_tail_split(native, rows256):
    """Routing built so that the down projection has 8 token blocks x 2 feature tiles of 256 rows
    over K = 4096: two tiles per XCD, each cut into 8 K slices whose sum the fix-up kernel scales
    (activation-row scale x weight-row scale x routed weight) and rounds."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd.layers.fused_moe import plan
    from fast_route_amd import _native as N
    _say("fp8 tail split")
    H, Fd, E, k, M = 512, 4096, 2, 1, 2048
    p = plan(M, H, Fd, E, k, torch.bfloat16, code=N.FR_FP8_E4M3)
    assert p.block == 256 and p.tail_bytes > 0 and p.split_k == 1
    g = torch.Generator().manual_seed(91)
    x = torch.randn(M, H, generator=g).bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.02).bfloat16()
    ids = torch.cat([torch.zeros(1280, dtype=torch.long), torch.ones(768, dtype=torch.long)])[torch.randperm(M, generator=g)]
    logits = torch.full((M, E), -4.0)
    logits[torch.arange(M), ids] = 4.0
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
    out = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
    torch.cuda.synchronize()
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_tiles_as_tall_as_the_experts_runs(native):
    """Runs that end one slot before, at and behind every unit of 32 rows, up to several tiles, and experts without a pair:
    the one-wavefront-per-SIMD kernel against the eight-wavefront kernels, bit for bit (same MFMAs, same order)."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say("fp8 tile heights")
    counts = [32 * u + d for u in range(1, 10) for d in (-1, 0, 1)] + [0, 320, 289, 575, 1060]
    H, Fd, E, M = 2048, 2048, len(counts), sum(counts)
    g = torch.Generator().manual_seed(95)
    x = torch.randn(M, H, generator=g).bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.02).bfloat16()
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(M, generator=g)]
    logits = torch.nn.functional.one_hot(ids, E).float() * 20.0
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
    res = []
    try:
        for no_quad in (False, True):
            with fr.tunables(block=256, no_quad=no_quad):
                res.append(fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), 1, True))
        torch.cuda.synchronize()
    finally:
        fr.reset_tunables()
    assert torch.isfinite(res[0].float()).all() and res[0].float().abs().max() > 0
    assert torch.equal(res[0], res[1]), "the two 256-row fp8 kernels differ"


def test_fp8_layer_leaves_the_heights_to_the_kernel(native, kernels_of):
    """A layer whose plan routes for 160 rows and whose runs suit the one-wavefront-per-SIMD kernel: both GEMMs take it."""
    from fast_route_amd import _native as N, fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd.layers.fused_moe import plan
    _say("fp8 plan of 160 rows, tiles as tall as the runs")
    M, H, Fd, E, k = 1250, 4096, 2048, 8, 2
    assert plan(M, H, Fd, E, k, None, code=N.FR_FP8_E4M3).block == 160
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=97)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    weights = prepare_weights_fp8(w1.cuda(), w2.cuda())
    args = [x.cuda(), *weights, logits.cuda()]
    out, names = kernels_of(lambda: fused_moe_fp8(*args, k, True))
    assert sum("moe_gemm_quad_kernel" in n for n in names) == 2, names
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_one_tile_per_expert_where_the_plan_has_two(native, kernels_of):
    """Runs of about five units, one tile each alone on its weight tile, where the plan's 160 rows cut them in two."""
    from fast_route_amd import _native as N, fused_moe_fp8, prepare_weights_fp8
    from fast_route_amd.layers.fused_moe import plan
    M, H, Fd, E, k = 645, 4096, 3328, 8, 2
    _say("fp8, one tile per expert")
    assert plan(M, H, Fd, E, k, None, code=N.FR_FP8_E4M3).block == 160
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=98)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    args = [x.cuda(), *prepare_weights_fp8(w1.cuda(), w2.cuda()), logits.cuda()]
    out, names = kernels_of(lambda: fused_moe_fp8(*args, k, True))
    assert sum("moe_gemm_quad_kernel" in n for n in names) == 2, names
    assert torch.equal(out, fused_moe_fp8(*args, k, True))
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_cut_tiles_of_nine_units(native):
    """Both GEMMs' last round cut along K with tiles of 9 units (9 experts of two tiles each, 32 and 16 feature tiles, 32 K
    tiles): the result differs from that of whole tiles by the order of fp32 sums (and the codes of activated rows that
    round the other way)."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say("fp8 cut tiles of nine units")
    H, Fd, E, M = 4096, 4096, 9, 9 * 545
    g = torch.Generator(device="cuda").manual_seed(98)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g, device="cuda") * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g, device="cuda") * 0.02).bfloat16()
    ids = torch.randperm(M, generator=g, device="cuda") % E
    logits = torch.nn.functional.one_hot(ids, E).float() * 20.0
    weights = prepare_weights_fp8(w1, w2)
    with fr.tunables(block=256, split_k=1):
        cut = fused_moe_fp8(x, *weights, logits, 1, True).float()
    with fr.tunables(block=256, split_k=1, no_tail_split=True):
        whole = fused_moe_fp8(x, *weights, logits, 1, True).float()
    assert torch.isfinite(cut).all() and not torch.equal(cut, whole), "nothing was cut"
    assert (cut - whole).norm() / whole.norm() <= 1e-2
    assert (cut - whole).abs().max() <= 2.0 ** -5 * whole.abs().max()


def test_fp8_one_wavefront_per_simd_tile_equals_the_eight_wavefront_tile(native):
    """fp8 on 256-row blocks with 16 K tiles (2048 elements) or more runs on four wavefronts of 128 x 128 outputs
    (moe_gemm_quad_kernel, 32x32x64 MFMAs); the no_quad knob sends the call to the eight-wavefront kernels.  Same
    MFMA shape and K order: equal bit for bit, and within the fp8 bounds of the oracle.  Sixteen experts with a mix
    of full, under-half and over-half blocks (half tiles), 2304 and 2560 elements of K (18 and 20 K tiles); top-2
    routing by logits."""
    import fast_route_amd as fr
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say("fp8 quad tile vs eight-wavefront tile")
    H, Fd, E, k, M = 2304, 2560, 16, 2, 2600
    g = torch.Generator().manual_seed(93)
    x = torch.randn(M, H, generator=g).bfloat16()
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.02).bfloat16()
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.02).bfloat16()
    logits = torch.randn(M, E, generator=g) + torch.linspace(2.0, -2.0, E)  # skewed loads: 1 .. 3 blocks per expert
    w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
    try:
        with fr.tunables(block=256):
            quad = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
        with fr.tunables(block=256, no_quad=True):
            eight = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
        torch.cuda.synchronize()
    finally:
        fr.reset_tunables()
    assert torch.equal(quad, eight), "the two 256-row fp8 kernels differ"
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = quad.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_fp8_random_shapes_against_oracle(native):
    """Sixteen seeded random fp8 layer shapes against the oracle (same tolerance as above)."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    rng = np.random.default_rng(8)
    for case in range(16):
        E = int(rng.choice([1, 2, 4, 8, 16, 64]))
        k = int(rng.integers(1, min(E, 6) + 1))
        H = int(rng.choice([256, 512, 1024, 4096]))
        Fd = int(rng.choice([256, 512, 768]))
        M = int(rng.choice([1, 2, 5, 17, 40, 100, 160, 257, 500]))
        _say(f"fp8 random case {case}: M={M} H={H} F={Fd} E={E} k={k}")
        x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=500 + case)
        x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
        w1q, w1s, w2q, w2s = prepare_weights_fp8(w1.cuda(), w2.cuda())
        out = fused_moe_fp8(x.cuda(), w1q, w1s, w2q, w2s, logits.cuda(), k, True)
        torch.cuda.synchronize()
        ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
        o = out.float().cpu()
        assert torch.isfinite(o).all()
        assert (o - ref).norm() / ref.norm() <= 1e-2, f"case {case}"
        assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max(), f"case {case}"


@pytest.mark.parametrize("H", [256, 8192, 8448, 16384, 16640])
@pytest.mark.parametrize("M", [1, 17])
def test_fp8_token_rows_of_the_routing_launch(native, H, M):
    """A small layer's token rows are quantised beside its routing: one chunk per thread of a workgroup, two, the last one partly
    filled, and beyond those a wavefront to a row.  Bounds as in test_fp8_layer_vs_oracle: 256 of 16640 elements left out or taken from
    the wrong place would be 12 % of the norm."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say(f"fp8 token rows H={H} M={M}")
    Fd, E, k = 256, 2, 1
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=79)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    out = fused_moe_fp8(x.cuda(), *prepare_weights_fp8(w1.cuda(), w2.cuda()), logits.cuda(), k, True)
    torch.cuda.synchronize()
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


@pytest.mark.parametrize("M,H", [(128, 1024), (128, 1280), (129, 1280), (129, 1792), (129, 2048), (513, 4096), (1024, 512), (1024, 2048)])
def test_fp8_token_rows_by_length_and_count(native, M, H):
    """Both sides of the rule that gives a token row beside the routing a wavefront or a workgroup: a wavefront to every row with the last
    workgroup partly filled, a workgroup to every row.  Bounds as in test_fp8_layer_vs_oracle."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    _say(f"fp8 token rows M={M} H={H}")
    Fd, E, k = 256, 2, 1
    x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=83)
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    out = fused_moe_fp8(x.cuda(), *prepare_weights_fp8(w1.cuda(), w2.cuda()), logits.cuda(), k, True)
    torch.cuda.synchronize()
    ref, _ = oracle.fused_moe_fp8(x, w1, w2, logits, k, True)
    o = out.float().cpu()
    assert torch.isfinite(o).all()
    assert (o - ref).norm() / ref.norm() <= 1e-2
    assert (o - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


@pytest.mark.parametrize("E,topk,Ms", [(32, 4, (128, 129, 250)), (32, 1, (256, 257, 511)), (64, 6, (64, 65, 129, 170)), (64, 1, (193, 256))])
def test_fp8_routing_passes_of_several_logits_per_lane(native, E, topk, Ms):
    """fp8 layers gate up to 1024 pairs in one workgroup: one to four passes of 128 (64) tokens with several logits per lane, wavefronts
    without a token in the last one.  The same logits at an address that vector loads cannot read take one per lane in the same launch:
    the outputs are bit-equal."""
    from fast_route_amd import fused_moe_fp8, prepare_weights_fp8
    H = Fd = 256
    for M in Ms:
        _say(f"fp8 routing passes E={E} k={topk} M={M}")
        x, logits, w1, w2 = oracle.make_inputs(M, H, Fd, E, seed=89 + M)
        args = (x.bfloat16().cuda(), *prepare_weights_fp8(w1.bfloat16().cuda(), w2.bfloat16().cuda()))
        buf = torch.empty(M * E + 1, device="cuda")
        outs = []
        for odd in (0, 1):
            dev = buf[odd:odd + M * E].view(M, E)
            dev.copy_(logits)
            outs.append(fused_moe_fp8(*args, dev, topk, True))
        assert torch.isfinite(outs[0].float()).all() and outs[0].abs().max() > 0
        assert torch.equal(outs[0], outs[1])
