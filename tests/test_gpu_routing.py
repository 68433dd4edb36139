"""GPU parity: block-aligned routing arrays, bit-exact against the CPU oracle."""
import sys

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _say(msg):
    print("[case] " + msg, flush=True)
    sys.stdout.flush()


def _check(ids: torch.Tensor, B: int, E: int):
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    s, e, npost = moe_align_block_size(ids.cuda(), B, E)
    torch.cuda.synchronize()
    rs, re_, rn = oracle.moe_align_block_size(ids, B, E)
    n = ids.numel()
    assert s.shape[0] == n + E * (B - 1) and e.shape[0] == n + E and s.dtype == torch.int32
    npost = int(npost.cpu()[0])
    assert npost == int(rn[0])
    assert np.array_equal(s.cpu().numpy(), rs), "sorted_token_ids differ"  # includes padding and tail == n
    assert np.array_equal(e.cpu().numpy()[: npost // B], re_[: npost // B]), "expert_ids differ"


def test_align_reference_docstring_example(native):
    _say("align docstring example")
    ids = torch.tensor([[2, 3, 4], [1, 2, 4], [1, 3, 4], [1, 2, 3]], dtype=torch.int32)
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    s, e, n = moe_align_block_size(ids.cuda(), 4, 5)
    assert s.cpu()[:16].tolist() == [3, 6, 9, 12, 0, 4, 10, 12, 1, 7, 11, 12, 2, 5, 8, 12]
    assert e.cpu()[:4].tolist() == [1, 2, 3, 4] and n.cpu().tolist() == [16]


@pytest.mark.parametrize("E,k", [(8, 2), (64, 6), (5, 3), (16, 1), (256, 8), (300, 4), (1024, 2)])
@pytest.mark.parametrize("B", [16, 32, 64, 128, 1, 4])
def test_align_small_and_ragged(native, E, k, B):
    for M in (0, 1, 7, 64, 333, 2500):
        _say(f"align E={E} k={k} B={B} M={M}")
        rng = np.random.default_rng(E * 7 + k * 3 + B + M)
        ids = rng.integers(0, E, size=(M, k)).astype(np.int32)
        if M > 3:
            ids[ids == E - 1] = 0  # an empty expert
        _check(torch.from_numpy(ids), B, E)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_align_all_to_one_expert_and_id_dtypes(native, dtype):
    _say(f"align single expert dtype={dtype}")
    ids = torch.full((1000, 2), 3, dtype=dtype)
    _check(ids, 64, 8)
    ids = torch.arange(4000, dtype=dtype).reshape(2000, 2) % 8
    _check(ids, 16, 8)


@pytest.mark.parametrize("B", [16, 32, 64, 128])
def test_align_routing_stress_config(native, B):
    """65536 tokens, 64 experts, top-6, Zipf(1.2)-skewed load: the multi-launch path."""
    _say(f"align stress B={B}")
    logits = oracle.zipf_logits(65536, 64, seed=2024)
    _, ids = oracle.gating_topk(logits, 6)
    counts = torch.bincount(ids.reshape(-1).long(), minlength=64)
    assert counts.max() > 8 * counts.min().clamp(min=1)  # really imbalanced
    _check(ids, B, 64)
    # also through int64 ids and after the GPU's own gating of the same logits
    from fast_route_amd.ops.stable_route import topk_softmax
    w = torch.empty((65536, 6), dtype=torch.float32, device="cuda")
    gi = torch.empty((65536, 6), dtype=torch.int32, device="cuda")
    topk_softmax(w, gi, None, logits.cuda(), renormalize=True)
    assert torch.equal(gi.cpu(), ids)
    _check(ids.long(), B, 64)


def test_align_medium_sizes_cross_path_boundary(native):
    for n_tokens in (1024, 1025, 1365, 1366, 2730, 2731, 8192, 20000):  # 6144 / 6150 pairs straddle the one-workgroup limit
        _say(f"align boundary M={n_tokens}")
        rng = np.random.default_rng(n_tokens)
        ids = rng.integers(0, 64, size=(n_tokens, 6)).astype(np.int32)
        _check(torch.from_numpy(ids), 32, 64)


@pytest.mark.parametrize("n,E", [(6145, 64), (6145, 1), (8193, 8), (262144, 64), (262145, 64), (524289, 8), (700001, 100), (300, 257),
                                 (32768, 512), (32769, 512), (131072, 512), (131073, 512)])
def test_align_segment_lengths_of_the_large_sort(native, n, E):
    """Batches beyond one workgroup: the first size, one pair into a new workgroup, the sizes up to which 64 experts keep one-round
    segments and from which long batches take longer ones, more experts than the one-workgroup form has, and 512 experts
    at the last sizes of one round per segment and of the two launches."""
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    _say(f"align n={n} E={E}")
    g = torch.Generator().manual_seed(n + E)
    p = (torch.arange(E) + 1.0) ** -1.2
    for B in (16, 160):
        ids = torch.multinomial(p, n, replacement=True, generator=g).int().view(n, 1)
        if E > 2:
            ids[ids == E // 2] = 0  # an expert without a pair
        s, e, npost = moe_align_block_size(ids.cuda(), B, E)
        rs, re_, rn = oracle.moe_align_block_size(ids, B, E)
        total = int(rn[0])
        assert int(npost.cpu()[0]) == total
        assert (s.cpu().numpy() == rs).all()
        assert (e.cpu().numpy()[: total // B] == re_[: total // B]).all()


@pytest.mark.parametrize("n,E", [(6145, 64), (0, 257), (1025, 300), (32768, 512), (131073, 512), (524289, 8), (5000, 600), (0, 1024)])
def test_align_stays_in_the_workspace_it_asks_for(native, n, E):
    """Two and three launches in a workspace of exactly the stated size: the result is the oracle's, the words behind it are untouched,
    and a byte less is refused."""
    from fast_route_amd import _native as N
    _say(f"align workspace n={n} E={E}")
    B, lib = 32, N.lib()
    ids = torch.randint(0, E, (n, 1), generator=torch.Generator().manual_seed(n + E)).int()
    need = lib.fr_moe_align_workspace_bytes(n, E)
    assert need > 0
    dev, ws = ids.cuda(), torch.full((need // 4 + 64,), -7, dtype=torch.int32, device="cuda")
    out = [torch.empty(k, dtype=torch.int32, device="cuda") for k in (n + E * (B - 1), n + E, 1)]
    call = lambda size: lib.fr_moe_align(dev.data_ptr() or None, N.FR_I32, n, E, B, *(t.data_ptr() for t in out), ws.data_ptr(), size, N.stream_ptr(dev.device))
    assert call(need - 1) != 0
    N.check(call(need))
    torch.cuda.synchronize()
    rs, re_, rn = oracle.moe_align_block_size(ids, B, E)
    total = int(rn[0])
    assert int(out[2]) == total and (out[0].cpu().numpy() == rs).all() and (out[1].cpu().numpy()[: total // B] == re_[: total // B]).all()
    assert (ws[need // 4:] == -7).all()


@pytest.mark.parametrize("n", [100, 20000])
@pytest.mark.parametrize("integer", [np.int64, np.int32, torch.tensor], ids=["int64", "int32", "tensor"])
def test_align_takes_any_integer(native, n, integer):
    """block_size and num_experts as numpy or torch integers, with and without scratch for the sort."""
    from fast_route_amd.ops.fused_moe import moe_align_block_size
    _say(f"align integers n={n} {integer}")
    ids = (torch.arange(n, dtype=torch.int32) * 7 % 64).view(n, 1).cuda()
    for got, want in zip(moe_align_block_size(ids, integer(32), integer(64)), moe_align_block_size(ids, 32, 64)):
        used = want.numel() if want.numel() != n + 64 else n // 32
        assert torch.equal(got[:used], want[:used])


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_align_returns_plain_tensors(native, dtype):
    """Ids of a torch.Tensor subclass: the routing arrays are plain tensors all the same."""
    from fast_route_amd.ops.fused_moe import moe_align_block_size

    class Ids(torch.Tensor):
        pass

    _say(f"align subclass {dtype}")
    for n in (100, 20000):
        ids = (torch.arange(n, dtype=dtype) * 7 % 64).view(n, 1).cuda()
        got, want = moe_align_block_size(ids.as_subclass(Ids), 32, 64), moe_align_block_size(ids, 32, 64)
        assert all(type(t) is torch.Tensor for t in got)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1][: n // 32], want[1][: n // 32]) and torch.equal(got[2], want[2])
