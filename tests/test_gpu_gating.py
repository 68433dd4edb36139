"""GPU parity: gating kernels vs the CPU oracle.  ids bit-exact, weights to 1e-6."""
import sys

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
W_ATOL = 2e-6  # fp32 softmax weights in [0, 1]: a few ulp of expf/divide


def _say(msg):
    print("[case] " + msg, flush=True)
    sys.stdout.flush()


def _run_gating(logits_dev, topk, renorm):
    from fast_route_amd.ops.stable_route import topk_softmax
    M = logits_dev.shape[0]
    w = torch.empty((M, topk), dtype=torch.float32, device="cuda")
    ids = torch.empty((M, topk), dtype=torch.int32, device="cuda")
    topk_softmax(w, ids, None, logits_dev, renormalize=renorm)
    torch.cuda.synchronize()
    return w.cpu(), ids.cpu()


@pytest.mark.parametrize("E,topk", [(8, 2), (16, 4), (64, 6), (1, 1), (3, 2), (5, 5), (24, 3), (100, 7), (256, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("renorm", [True, False])
def test_gating_parity(native, E, topk, dtype, renorm):
    for M in (1, 63, 1000, 2500):
        _say(f"gating E={E} k={topk} dtype={dtype} renorm={renorm} M={M}")
        g = torch.Generator().manual_seed(E * 131 + topk * 7 + M)
        logits = torch.randn(M, E, generator=g).to(dtype)  # bf16/fp16 rounding creates exact ties
        w, ids = _run_gating(logits.cuda(), topk, renorm)
        rw, rid = oracle.gating_topk(logits, topk, renorm)
        assert torch.equal(ids, rid), "gating ids differ"
        torch.testing.assert_close(w, rw, atol=W_ATOL, rtol=0)


def test_gating_ties_and_special_rows(native):
    _say("gating special rows")
    rows = [
        [0.0] * 8,                                   # all equal -> ids 0..k-1
        [1.0, 3.0, 3.0, 0.0, 3.0, 1.0, 1.0, -2.0],   # three-way tie
        [-30.0, -30.0, -30.0, -30.0, -30.0, 30.0, -30.0, -30.0],
        [5.0, 4.0, 3.0, 2.0, 1.0, 0.0, -1.0, -2.0],
        [-2.0, -1.0, 0.0, 1.0, 2.0, 3.0, 4.0, 5.0],
        [-0.0, 0.0, -0.0, 0.0, -1.0, 0.0, -0.0, -1.0],  # signed zeros are one value: ties by index
    ]
    logits = torch.tensor(rows)
    for k in (1, 2, 4, 8):
        for renorm in (True, False):
            w, ids = _run_gating(logits.cuda(), k, renorm)
            rw, rid = oracle.gating_topk(logits, k, renorm)
            assert torch.equal(ids, rid)
            torch.testing.assert_close(w, rw, atol=W_ATOL, rtol=0)
    w, ids = _run_gating(logits.cuda(), 4, True)
    assert ids[0].tolist() == [0, 1, 2, 3] and ids[1].tolist() == [1, 2, 4, 0]


@pytest.mark.parametrize("E,topk", [(32, 5), (64, 6), (64, 16), (64, 40), (128, 8), (256, 8), (48, 3)])
def test_gating_ties_many_experts(native, E, topk):
    """Rows built from a handful of distinct values, so every round of the selection has
    ties inside a lane, across lanes and across the vectors of a lane; +0 / -0 tie too.
    (topk = 40 exceeds the result slots of the few-lanes-per-token form: fallback path.)"""
    _say(f"gating ties E={E} topk={topk}")
    g = torch.Generator().manual_seed(E * 131 + topk)
    vals = torch.tensor([0.0, -0.0, 1.5, -1.5, 3.0, 0.25])
    logits = vals[torch.randint(0, len(vals), (1300, E), generator=g)]  # long enough for the few-lanes-per-token form
    logits[0] = 0.0
    logits[1] = torch.arange(E, dtype=torch.float32) % 3
    logits[2] = -torch.arange(E, dtype=torch.float32)
    for renorm in (True, False):
        w, ids = _run_gating(logits.cuda(), topk, renorm)
        rw, rid = oracle.gating_topk(logits, topk, renorm)
        assert torch.equal(ids, rid)
        torch.testing.assert_close(w, rw, atol=W_ATOL, rtol=0)
    # a row stride that is not a multiple of 4 takes the one-logit-per-lane path
    wide = torch.zeros(1300, E + 3)
    wide[:, :E] = logits
    w2, ids2 = _run_gating(wide.cuda()[:, :E], topk, True)
    assert torch.equal(ids2, oracle.gating_topk(logits, topk, True)[1])


@pytest.mark.parametrize("E,topk", [(20, 3), (32, 16), (64, 6), (64, 15), (128, 8), (256, 32)])
def test_gating_near_ties_many_experts(native, E, topk):
    """fp32 logits a few units in the last place apart: the few-lanes-per-token form packs the expert index into the low
    bits of its keys and has to notice that such neighbours need the exact ones.  Rows of clear-cut logits share the
    wavefronts; masked experts (-inf) tie among themselves."""
    _say(f"gating near ties E={E} topk={topk}")
    g = torch.Generator().manual_seed(E * 17 + topk)
    for sign in (1.0, -1.0):
        logits = sign * (1.0 + torch.randint(0, 70, (1300, E), generator=g).float() * 2.0 ** -23)
        logits[::3] = torch.randn(logits[::3].shape, generator=g)
        logits[1::7] = logits[1::7] * (1 + 2.0 ** -20 * torch.randn(logits[1::7].shape, generator=g))
        logits[2::5, topk:] = float("-inf")
        for renorm in (True, False):
            w, ids = _run_gating(logits.cuda(), topk, renorm)
            rw, rid = oracle.gating_topk(logits, topk, renorm)
            assert torch.equal(ids, rid)
            torch.testing.assert_close(w, rw, atol=W_ATOL, rtol=0)


@pytest.mark.parametrize("E,topk", [(20, 16), (32, 5), (64, 1), (64, 6), (64, 16), (128, 8), (128, 32), (252, 9), (256, 8), (256, 64)])
@pytest.mark.parametrize("spread", [2, 40, 700, 20000])
def test_gating_packed_key_classes(native, E, topk, spread):
    """fp32 logits that share the upper bits of their packed keys in every way: classes that end with the last winner or
    reach beyond it, several classes in one row, exact duplicates with low bits set (16-bit logits scaled in fp32), masked
    experts.  `spread` is the width of a row's logits in units in the last place."""
    _say(f"gating classes E={E} topk={topk} spread={spread}")
    g = torch.Generator().manual_seed(E * 31 + topk * 7 + spread)
    for sign in (1.0, -1.0):
        logits = sign * (1.0 + torch.randint(0, spread, (1100, E), generator=g).float() * 2.0 ** -23)
        logits[1::5] = torch.randn(logits[1::5].shape, generator=g).bfloat16().float() * 0.37
        logits[2::5, max(topk - 1, 1):] = float("-inf")
        logits[3::5, ::3] += torch.randint(0, 3, logits[3::5, ::3].shape, generator=g).float()
        for renorm in (True, False):
            w, ids = _run_gating(logits.cuda(), topk, renorm)
            rw, rid = oracle.gating_topk(logits, topk, renorm)
            assert torch.equal(ids, rid)
            torch.testing.assert_close(w, rw, atol=W_ATOL, rtol=0)


@pytest.mark.parametrize("E,topk", [(32, 4), (64, 6), (128, 8), (256, 8)])
def test_gating_nan_and_infinite_rows_many_experts(native, E, topk):
    """Rows with NaN or +inf next to ordinary ones: NaN orders above +inf (the order of the keys), such a row's weights are
    NaN, and the other rows of its wavefront are what they are without it."""
    _say(f"gating nan / inf rows E={E} topk={topk}")
    g = torch.Generator().manual_seed(E + topk)
    logits = torch.randn(1200, E, generator=g)
    logits[::7, E // 3] = float("nan")
    logits[3::11, E - 1] = float("inf")
    logits[::14, 1] = float("nan")
    bad = (logits.isnan() | (logits == float("inf"))).any(dim=1)
    masked = ~bad & (torch.arange(1200) % 5 == 0)
    logits[masked, topk // 2:] = float("-inf")
    lifted = torch.where(logits.isnan(), 9e30, torch.where(logits == float("inf"), 8e30, logits))
    for renorm in (True, False):
        w, ids = _run_gating(logits.cuda(), topk, renorm)
        rw, rid = oracle.gating_topk(lifted, topk, renorm)
        assert torch.equal(ids, rid)
        assert w[bad].isnan().all()
        torch.testing.assert_close(w[~bad], rw[~bad], atol=W_ATOL, rtol=0)


def test_gating_reference_route_test_recipe(native):
    """tests/test_route.py:12-77 of the reference: weights vs topk(softmax(h@gate)), atol 1e-2."""
    for seed in range(3):
        for m, topk in ((128, 2), (512, 4)):
            _say(f"route recipe seed={seed} m={m} topk={topk}")
            torch.manual_seed(seed)
            h = (torch.randn((m, 4096)) / 10).half()
            gate = (torch.randn((4096, 16)) / 10).half()
            from fast_route_amd.ops.stable_route import fused_route
            tw = torch.empty(m, 16, dtype=torch.float32, device="cuda")
            ti = torch.empty(m, 16, dtype=torch.int32, device="cuda")
            w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
            torch.cuda.synchronize()
            score = h.float() @ gate.float()
            rw, rid = torch.topk(torch.softmax(score, -1), topk)
            rw = rw / rw.sum(-1, keepdim=True)
            torch.testing.assert_close(w.cpu(), rw, atol=1e-2, rtol=0)
            ow, oid = oracle.route_from_gate(h, gate, topk)
            torch.testing.assert_close(w.cpu(), ow, atol=1e-4, rtol=0)
            # ids can only differ where fp32 accumulation order flips a near-tie
            assert (ids.cpu() != oid).float().mean() < 0.01


@pytest.mark.parametrize("E,topk,H", [(8, 2, 1024), (64, 6, 2048), (16, 4, 520), (5, 2, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_route_gate_fused_gemm(native, E, topk, H, dtype):
    from fast_route_amd.ops.stable_route import fused_route
    for M in (1, 70, 300):
        _say(f"route_gate E={E} k={topk} H={H} dtype={dtype} M={M}")
        g = torch.Generator().manual_seed(E + H + M)
        h = (torch.randn(M, H, generator=g) / 4).to(dtype)
        gate = (torch.randn(H, E, generator=g) / 4).to(dtype)
        tw = torch.empty(M, topk, dtype=torch.float32, device="cuda")
        ti = torch.empty(M, topk, dtype=torch.int32, device="cuda")
        w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
        torch.cuda.synchronize()
        logits = h.double() @ gate.double()
        ow, oid = oracle.gating_topk(logits.float(), topk, True)
        # fp32 MFMA accumulation vs float64 reference: ids may flip only at near-ties
        flips = (ids.cpu() != oid)
        assert flips.float().mean() < 0.02
        ok = ~flips.any(dim=1)
        torch.testing.assert_close(w.cpu()[ok], ow[ok], atol=1e-4, rtol=0)


@pytest.mark.parametrize("E,topk,H", [(16, 2, 2056), (3, 1, 1032), (9, 3, 4088)])
@pytest.mark.parametrize("M", [17, 4096, 4097])
def test_route_gate_sixteen_wavefronts(native, E, topk, H, M):
    """Up to 16 experts and 4096 tokens a workgroup's sixteen wavefronts split chunks of 1024 K rows: a last chunk of a few rows,
    a wavefront's share of it empty, a ragged last workgroup, and the batch size where the form changes."""
    from fast_route_amd.ops.stable_route import fused_route
    _say(f"route_gate E={E} H={H} M={M}")
    g = torch.Generator().manual_seed(E * 7 + H)
    h = (torch.randn(M, H, generator=g) / 4).to(torch.float16)
    gate = (torch.randn(H, E, generator=g) / 4).to(torch.float16)
    tw = torch.empty(M, topk, dtype=torch.float32, device="cuda")
    ti = torch.empty(M, topk, dtype=torch.int32, device="cuda")
    w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
    torch.cuda.synchronize()
    ow, oid = oracle.gating_topk((h.double() @ gate.double()).float(), topk, True)
    flips = (ids.cpu() != oid)
    assert flips.float().mean() < 0.002  # near-ties of fp32 sums
    ok = ~flips.any(dim=1)
    torch.testing.assert_close(w.cpu()[ok], ow[ok], atol=1e-4, rtol=0)


@pytest.mark.parametrize("E,topk,H", [(8, 2, 264), (64, 6, 256), (24, 3, 512), (128, 8, 256), (100, 6, 512)])
def test_route_gate_large_batch(native, E, topk, H):
    """From 16384 tokens on the kernel takes its unsplit form (64 or 128 tokens per workgroup,
    every wavefront the whole K range of its own tokens); 16500 tokens leave a ragged last
    workgroup."""
    from fast_route_amd.ops.stable_route import fused_route
    M = 16500
    _say(f"route_gate large batch E={E} k={topk} H={H}")
    g = torch.Generator().manual_seed(E * 7 + H)
    h = (torch.randn(M, H, generator=g) / 4).to(torch.bfloat16)
    gate = (torch.randn(H, E, generator=g) / 4).to(torch.bfloat16)
    tw = torch.empty(M, topk, dtype=torch.float32, device="cuda")
    ti = torch.empty(M, topk, dtype=torch.int32, device="cuda")
    w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
    torch.cuda.synchronize()
    ow, oid = oracle.gating_topk((h.double() @ gate.double()).float(), topk, True)
    flips = (ids.cpu() != oid)
    assert flips.float().mean() < 0.02
    ok = ~flips.any(dim=1)
    torch.testing.assert_close(w.cpu()[ok], ow[ok], atol=1e-4, rtol=0)


@pytest.mark.parametrize("E,topk,H", [(16, 2, 4096), (128, 4, 1024), (100, 3, 512)])
def test_fused_route_half_and_int64_buffers(native, E, topk, H):
    """The reference's own recipe hands fused_route fp16 weight and int64 id buffers of [M, E]
    (tests/test_route.py:30-38) and allows up to 128 experts (ops/stable_route.py:130-134):
    both must give the fp32-logit result, not one rounded to the operand type first."""
    from fast_route_amd.ops.stable_route import fused_route
    for M in (3, 257):
        _say(f"fused_route fp16/int64 buffers E={E} k={topk} H={H} M={M}")
        g = torch.Generator().manual_seed(E * 31 + H + M)
        h = (torch.randn(M, H, generator=g) / 10).half()
        gate = (torch.randn(H, E, generator=g) / 10).half()
        tw = torch.empty(M, E, dtype=torch.float16, device="cuda")
        ti = torch.empty(M, E, dtype=torch.int64, device="cuda")
        w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
        torch.cuda.synchronize()
        assert w.dtype == torch.float16 and ids.dtype == torch.int64 and w.shape == ids.shape == (M, topk)
        ow, oid = oracle.gating_topk((h.double() @ gate.double()).float(), topk, True)
        flips = (ids.cpu() != oid.long())
        assert flips.float().mean() < 0.02   # fp32 against float64 logits: near-ties only
        ok = ~flips.any(dim=1)
        torch.testing.assert_close(w.cpu().float()[ok], ow[ok], atol=1e-3, rtol=0)  # fp16 storage of the weights


@pytest.mark.parametrize("E,topk", [(20, 3), (32, 4), (32, 20), (36, 6), (64, 1), (64, 6), (64, 17), (68, 2), (256, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_launch_routing_is_the_separate_launches(native, E, topk, dtype):
    """Small layers gate and sort in one launch, with several logits per lane for 17 to 64 experts; the layer is then bit
    for bit that of the gating launch's ids and weights.  Token counts at the edges of the wavefronts' groups, of the one
    launch and beyond it; rows of ties, of logits that differ below the packed keys, of infinities and NaN; logits that
    vector loads cannot read and weights that are not renormalised, which take the other form."""
    from fast_route_amd import fused_experts, fused_moe
    H = Fd = 128
    g = torch.Generator().manual_seed(E * 7 + topk)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.05).bfloat16().cuda()
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.05).bfloat16().cuda()
    for M in (1, 3, 4, 15, 17, 63, 64, 65, 129):
        x = torch.randn(M, H, generator=g).bfloat16().cuda()
        noise = torch.randn(M, E, generator=g)
        rows = {"random": noise, "ties": (noise * 2).round(), "near": 1.0 + noise * 2.0 ** -22,
                "masked": torch.where(torch.rand(M, E, generator=g) < 0.5, noise, torch.tensor(-float("inf")))}
        rows["nan"] = torch.where(torch.rand(M, E, generator=g) < 0.05, torch.tensor(float("nan")), noise)
        for name, logits in rows.items():
            for renorm in (True, False):
                for odd in (False, True):
                    if (odd or not renorm) and name not in ("random", "ties"):
                        continue
                    _say(f"one-launch routing E={E} k={topk} {dtype} M={M} {name} renorm={renorm} odd={odd}")
                    buf = torch.empty(M * E + 1, dtype=dtype, device="cuda")
                    dev = buf[int(odd):int(odd) + M * E].view(M, E)
                    dev.copy_(logits)
                    w, ids = _run_gating(dev, topk, renorm)
                    out = fused_moe(x, w1, w2, dev, topk, renorm)
                    ref = fused_experts(x, w1, w2, w.cuda(), ids.cuda())
                    assert torch.equal(out.isnan(), ref.isnan()), "other rows are NaN"
                    assert torch.equal(out.nan_to_num(), ref.nan_to_num()), "layer differs"


@pytest.mark.parametrize("E,topk", [(8, 2), (16, 2)])
@pytest.mark.parametrize("H", [1024, 1032, 4096, 4104, 9224])
def test_route_gate_chunks_asked_for_together(native, E, topk, H):
    """Experts in whole groups of 8: four chunks of 1024 K rows are loaded ahead.  One chunk, a chunk and a few rows, four
    chunks, a second set of a few rows, a set that ends in its second chunk; a ragged last workgroup."""
    from fast_route_amd.ops.stable_route import fused_route
    for M in (1, 33):
        _say(f"route_gate chunks E={E} H={H} M={M}")
        g = torch.Generator().manual_seed(E * 7 + H)
        h = (torch.randn(M, H, generator=g) / 4).to(torch.float16)
        gate = (torch.randn(H, E, generator=g) / 4).to(torch.float16)
        tw = torch.empty(M, topk, dtype=torch.float32, device="cuda")
        ti = torch.empty(M, topk, dtype=torch.int32, device="cuda")
        w, ids = fused_route(h.cuda(), gate.cuda(), topk, tw, ti, True)
        torch.cuda.synchronize()
        logits = h.double() @ gate.double()
        ow, oid = oracle.gating_topk(logits.float(), topk, True)
        # fp32 sums of 9224 products of spread 1/16 stay within 1e-4 of the exact ones: ids may differ at closer ties only
        top = torch.sort(logits, dim=1, descending=True).values
        clear = (top[:, :topk] - top[:, 1:topk + 1]).min(dim=1).values > 2e-4
        assert clear.float().mean() > 0.9
        assert torch.equal(ids.cpu()[clear], oid[clear])
        torch.testing.assert_close(w.cpu()[clear], ow[clear], atol=1e-4, rtol=0)


@pytest.mark.parametrize("E,M,H,together", [(16, 128, 1032, 4), (16, 129, 1032, 1), (16, 2048, 4104, 1), (16, 2049, 2048, 4), (16, 128, 1024, 1), (8, 129, 4096, 4),
                                            (8, 2048, 1032, 4), (12, 129, 4096, 1), (5, 129, 4096, 4)])
def test_route_gate_chunks_by_experts_and_tokens(native, kernels_of, E, M, H, together):
    """Where four chunks of gate rows are asked for together and where one: both sides of the rule, against float64 logits.  Bounds as in
    test_route_gate_chunks_asked_for_together."""
    import re
    from fast_route_amd.ops.stable_route import fused_route
    _say(f"route_gate chunks E={E} M={M} H={H}")
    g, k = torch.Generator().manual_seed(E * 7 + M), 2
    h = (torch.randn(M, H, generator=g) / 4).to(torch.float16)
    gate = (torch.randn(H, E, generator=g) / 4).to(torch.float16)
    tw, ti = torch.empty(M, k, dtype=torch.float32, device="cuda"), torch.empty(M, k, dtype=torch.int32, device="cuda")
    (w, ids), names = kernels_of(lambda: fused_route(h.cuda(), gate.cuda(), k, tw, ti, True))
    used = [n for n in names if "route_gate_kernel" in n]
    assert len(used) == 1 and re.search(r"Li16ELi%dEE|, 16, %d>" % (together, together), used[0]), names
    logits = h.double() @ gate.double()
    ow, oid = oracle.gating_topk(logits.float(), k, True)
    top = torch.sort(logits, dim=1, descending=True).values
    clear = (top[:, :k] - top[:, 1:k + 1]).min(dim=1).values > 2e-4
    assert clear.float().mean() > 0.9
    assert torch.equal(ids.cpu()[clear], oid[clear])
    torch.testing.assert_close(w.cpu()[clear], ow[clear], atol=1e-4, rtol=0)


@pytest.mark.parametrize("E,topk,Ms", [(64, 6, (31, 32, 33)), (64, 2, (32, 33, 48, 49)), (36, 6, (32, 33)), (32, 4, (32, 33, 64, 65)), (20, 1, (65, 96, 97))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_one_launch_routing_at_its_last_sizes(native, E, topk, Ms, dtype):
    """The last token counts of the one launch, the first of two, and more than one pass of the one workgroup; rows with +inf, with
    both infinities, of -inf alone, masked with the type's lowest value, and with NaN.  Bit for bit the separate launches' layer."""
    from fast_route_amd import fused_experts, fused_moe
    H = Fd = 128
    g = torch.Generator().manual_seed(E * 11 + topk)
    w1 = (torch.randn(E, 2 * Fd, H, generator=g) * 0.05).bfloat16().cuda()
    w2 = (torch.randn(E, H, Fd, generator=g) * 0.05).bfloat16().cuda()
    for M in Ms:
        x = torch.randn(M, H, generator=g).bfloat16().cuda()
        noise, u = torch.randn(M, E, generator=g), torch.rand(M, E, generator=g)
        inf, lowest = torch.tensor(float("inf")), torch.tensor(torch.finfo(dtype).min)
        rows = {"random": noise, "+inf": torch.where(u < 0.03, inf, noise), "both": torch.where(u < 0.03, inf, torch.where(u > 0.6, -inf, noise)),
                "lowest": torch.where(u < 0.95, lowest, noise), "nan": torch.where(u < 0.03, torch.tensor(float("nan")), noise)}
        rows["-inf"] = torch.where(torch.arange(M)[:, None] % 3 == 0, -inf, noise)
        for name, logits in rows.items():
            _say(f"one-launch routing at its last sizes E={E} k={topk} {dtype} M={M} {name}")
            dev = logits.to(dtype).cuda()
            w, ids = _run_gating(dev, topk, True)
            out, ref = fused_moe(x, w1, w2, dev, topk, True), fused_experts(x, w1, w2, w.cuda(), ids.cuda())
            assert torch.equal(out.isnan(), ref.isnan()), "other rows are NaN"
            assert torch.equal(out.nan_to_num(), ref.nan_to_num()), "layer differs"
