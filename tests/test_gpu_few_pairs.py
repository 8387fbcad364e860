"""The layer call in 16-row blocks with bf16 activations, or with MXFP4 ones and few rows per expert (kernels of its own, without a sort up to 64 or 128
pairs and without a reduction where pairs rarely share an expert), against the step-by-step path.  With bf16 activations the arithmetic
and its order are the same; with MXFP4 ones the sums of such data are exact in any order: the same bits.  Data whose block scales lie far
apart are compared within the rounding of two orders of summation."""
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


def _poison(T, k, E, H, I, method, rows=16):
    """the memory that the next call of these (padded) sizes gets as its workspace holds NaNs, in bf16 and in fp32"""
    import sys
    plan = sys.modules["pyhip_amd.fused_moe"]._plan
    x = torch.empty(plan(T, k, E, H, I, method, rows)[2], dtype=torch.uint8, device="cuda")
    x.fill_(255)


@pytest.mark.parametrize("T,k,E,H,I,splitk", [
    (1, 1, 8, 512, 512, 0),          # one pair; every K split has one K-step
    (1, 4, 20, 1024, 2560, 0),       # a token's slots on four groups of waves, an uneven share of K-steps
    (1, 4, 8, 9216, 512, 0),         # four row groups to a workgroup, a K-step for each wave
    (1, 5, 8, 5632, 1536, 0),        # two
    (1, 6, 64, 512, 1024, 0),        # one; three slots for each group of waves
    (1, 9, 16, 512, 512, 0),         # more slots than the summing kernel holds
    (4, 1, 32, 512, 512, 0),         # summed by token
    (4, 8, 256, 512, 512, 4),        # the most pairs that are summed by token in 256 experts
    (5, 8, 256, 512, 512, 0),        # one token more
    (64, 1, 8, 512, 512, 0),         # 64 pairs in 8 experts
    (63, 1, 3, 512, 1024, 0),        # more than a block for an expert; an expert count that is no power of two
    (64, 1, 1, 512, 512, 1),         # one expert, four full blocks, no K split
    (8, 8, 16, 1024, 1536, 1),
    (65, 1, 8, 512, 512, 0),         # one pair more: two to a lane
    (13, 5, 8, 1536, 512, 0),        # an odd top-k
    (64, 2, 8, 1024, 512, 0),        # 128 pairs
    (128, 1, 12, 512, 1024, 1),
    (16, 8, 40, 512, 512, 0),        # as many workgroups as run at once
    (16, 8, 41, 512, 512, 0),        # more: sorted
    (129, 1, 33, 512, 512, 0),       # a pair more: sorted
    (10, 8, 640, 512, 512, 0),       # summed by token, more than 64 pairs
    (40, 4, 16, 512, 1536, 1),       # sorted, no K split
    (17, 4, 17, 1024, 1536, 0),      # sorted, four rows per expert
    (23, 3, 17, 512, 512, 0),        # one pair more
    (96, 8, 192, 512, 512, 0),       # sorted, several blocks for an expert
    (1, 2, 8, 512, 1024, 1),         # a top-2 token whose slots the reduction sums
])
@pytest.mark.parametrize("method", ["w4a16", "a4w4"])
def test_few_pairs_equal_the_stages(T, k, E, H, I, splitk, method):
    _equal_the_stages(T, k, E, H, I, splitk, method, 16)


@pytest.mark.parametrize("T,k,E,H,I,rows", [
    (1, 1, 8, 512, 512, 32),             # one row
    (72, 2, 9, 1024, 1536, 32),          # sixteen rows per expert: the most in fewer than 32
    (73, 2, 9, 512, 512, 32),            # more
    (40, 8, 40, 1536, 1024, 32),
    (150, 6, 75, 512, 512, 32),          # twelve: the most in 32 experts and more
    (90, 8, 192, 2560, 512, 32),         # an uneven share of K-steps
    (128, 1, 8, 512, 512, 32),           # 32 rows asked for, blocks of 16 found without a sort
    (140, 1, 9, 512, 512, 32),           # one K-step for each wave
    (72, 1, 3, 1024, 1536, 64),          # 24: the most in fewer than 32
    (49, 2, 4, 512, 512, 64),            # more
    (120, 3, 30, 1536, 512, 64),
    (96, 8, 64, 512, 1024, 64),          # twelve
])
def test_several_row_tiles_equal_the_stages(T, k, E, H, I, rows):
    _equal_the_stages(T, k, E, H, I, 0, "a4w4", rows)


def _equal_the_stages(T, k, E, H, I, splitk, method, rows):
    """plain routing, holes in it, no bias, an expert mask, a local token count, one expert; SiLU to bf16 and SwiGLU to fp32"""
    from pyhip_amd import fused_moe
    from pyhip_amd.enums import ActivationType
    L = cases.make_layer("", T, seed=T * 7 + k, bias=True, E=E, k=min(k, E), H=H, I=I, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    g = torch.Generator().manual_seed(T + E)
    ids = torch.from_numpy(L.topk_ids).clone()
    if E > 1:
        ids[0, 0] = ids[-1, -1]                       # an expert that two pairs share, also inside one token
    hole = ids.clone()
    hole[torch.rand(hole.shape, generator=g) < 0.3] = -1
    hole[T // 2] = E                                  # a token that nobody serves
    local = torch.tensor([T - 1], dtype=torch.int32, device="cuda")
    mask = (torch.rand(E, generator=g) < 0.6).to(torch.int32)
    mask[int(ids[0, 0])] = 1
    keep = mask.bool().cuda()
    s1, s2, b1, b2 = w1s.view(E, -1), w2s.view(E, -1), L.bias1.cuda() * 20, L.bias2.cuda() * 20
    ma, mb = w1[keep].contiguous(), w2[keep].contiguous()
    ma.is_shuffled = mb.is_shuffled = True
    rank = dict(w1_scale=s1[keep].reshape(-1, w1s.shape[-1]).contiguous(), w2_scale=s2[keep].reshape(-1, w2s.shape[-1]).contiguous(),
                bias1=b1[keep], bias2=b2[keep], expert_mask=mask.cuda())
    whole = dict(w1_scale=w1s, w2_scale=w2s, bias1=b1, bias2=b2)
    hidden, tw = L.hidden.cuda(), torch.from_numpy(L.topk_w).cuda()
    for name, wa, wb, t, kw in (("plain", w1, w2, ids, whole), ("holes", w1, w2, hole, whole),
                                ("no bias", w1, w2, ids, dict(whole, bias1=None, bias2=None)),
                                ("mask", ma, mb, ids, rank), ("local", w1, w2, ids, dict(whole, num_local_tokens=local)),
                                ("one expert", w1, w2, torch.full_like(ids, E - 1), whole)):      # full blocks, and one of 1 to 4 row tiles
        for more in (dict(), dict(dtype=torch.float32, activation=ActivationType.Swiglu)):
            print(f"few pairs T={T} k={L.k} E={E} H={H} I={I} {name} {sorted(more)}", flush=True)
            kw2 = dict(kw, method=method, block_size_M=rows, splitk=splitk, **more)
            want = fused_moe(hidden, wa, wb, tw, t.cuda(), return_parts=True, **kw2)[0]
            for _ in range(2):
                _poison(T, L.k, E, H, I, method, rows)
                got = fused_moe(hidden, wa, wb, tw, t.cuda(), **kw2)
                assert torch.equal(got, want)


@pytest.mark.parametrize("T,H,I", [(1, 544, 544), (1, 544, 8224), (3, 1440, 1440), (1, 992, 32 * 47), (20, 1440, 1056), (30, 576, 1440), (50, 1440, 1056)])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("method,rows", [("w4a16", 16), ("a4w4", 16), ("a4w4", 32), ("a4w4", 64)])
def test_few_pairs_leave_padding_alone(T, H, I, wide, method, rows):
    """Padded layers, activations at the true or the padded width.  The weights' padding is told, so it is not read: its rows and
    columns are filled with ones here, and what the padded columns of the activations hold does not matter either."""
    from pyhip_amd import fused_moe
    L = cases.make_layer("", T, seed=H, bias=True, E=32, k=2, H=H, I=I, router="softmax")
    w1, w1s, w2, w2s, b1, b2, hp, ip = cases.padded_device_weights(L)
    tw, ti = torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda()
    kw = dict(bias1=b1, bias2=b2, method=method, block_size_M=rows)
    x = torch.nn.functional.pad(L.hidden.cuda(), (0, hp))
    want = fused_moe(x, w1, w2, tw, ti, w1_scale=w1s, w2_scale=w2s, return_parts=True, **kw)[0]
    # ones (code 2) in the padding rows of w2, in whole row groups of 16, and in the padding columns of both, in whole 1 KB blocks' groups of 32
    f1, f2 = w1.clone(), w2.clone()
    v1 = f1.view(32, -1, f1.shape[2] // 64, 4, 16, 16)      # [E, N / 16, K / 128, group of 32, row, byte]
    v2 = f2.view(32, -1, f2.shape[2] // 64, 4, 16, 16)
    for v, real in ((v1, H), (v2, I)):
        for c in range(real, v.shape[2] * 128, 32):
            v[:, :, c // 128, c % 128 // 32] = 0x22
    f1.is_shuffled = f2.is_shuffled = True
    if wide:
        x[:, H:] = float("nan")
    else:
        x = x[:, :H]
        x = torch.nn.functional.pad(x, (0, 8), value=float("nan"))[:, :H]
    print("few pairs, padded", T, H, I, wide, flush=True)
    _poison(T, 2, 32, H + hp, I + ip, method, rows)
    got = fused_moe(x, f1, f2, tw, ti, w1_scale=w1s, w2_scale=w2s, hidden_pad=hp, intermediate_pad=ip, **kw)
    assert torch.equal(got[:, :H], want[:, :H]) and (not wide or (got[:, H:] == 0).all())


@pytest.mark.parametrize("T", [1, 4, 8, 9, 40])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("method,rows", [("w4a16", 16), ("a4w4", 16), ("a4w4", 32), ("a4w4", 64)])
def test_few_pairs_with_the_router(T, grouped, method, rows):
    from pyhip_amd import fused_moe, fused_moe_routed
    L = cases.make_layer("", T, seed=T, E=256, k=8, H=512, I=512, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    logits = torch.randn(T, 256, generator=torch.Generator().manual_seed(T)).cuda()
    kw = dict(w1_scale=w1s, w2_scale=w2s, method=method, block_size_M=rows)
    print("few pairs, routed", T, grouped, flush=True)
    out, tw, ti = fused_moe_routed(L.hidden.cuda(), w1, w2, logits, 8, return_routing=True,
                                   **(dict(num_expert_group=8, topk_group=4) if grouped else {}), **kw)
    want = fused_moe(L.hidden.cuda(), w1, w2, tw, ti, return_parts=True, **kw)[0]
    assert torch.equal(out, want)


@pytest.mark.parametrize("T,k,method,rows", [(2, 1, "w4a16", 16), (1, 3, "w4a16", 16), (12, 1, "w4a16", 16), (12, 1, "a4w4", 16), (100, 1, "a4w4", 32),
                                             (100, 1, "a4w4", 64)])
def test_mask_with_more_entries_than_matrices(T, k, method, rows):
    """Not a call that means anything, but one that reads nothing past the weights: pairs whose number among the mask's entries is no matrix
    are left out, and the tokens of the others have their results."""
    from pyhip_amd import fused_moe
    E, here = 48, 24
    L = cases.make_layer("", T, seed=T, E=E, k=k, H=512, I=512, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(0, here, (T, k), generator=g, dtype=torch.int32)
    ids[0] = torch.arange(E - k, E)                     # a token whose experts are all past the matrices
    if T > 2:
        ids[T - 1] = here                               # the first of them
    tw = torch.rand(T, k, generator=g).cuda()
    want = fused_moe(L.hidden.cuda(), w1, w2, tw, ids.cuda(), w1_scale=w1s, w2_scale=w2s, method=method, block_size_M=rows)
    half = lambda w: w.view(E, -1)[:here].reshape(-1, w.shape[-1]).contiguous()
    ma, mb = w1[:here].contiguous(), w2[:here].contiguous()
    ma.is_shuffled = mb.is_shuffled = True
    print("few pairs, wide mask", T, k, method, rows, flush=True)
    got = fused_moe(L.hidden.cuda(), ma, mb, tw, ids.cuda(), w1_scale=half(w1s), w2_scale=half(w2s), method=method, block_size_M=rows,
                    expert_mask=torch.ones(E, dtype=torch.int32, device="cuda"))
    held = (ids < here).all(dim=1).cuda()
    assert held.sum() == T - (1 if T <= 2 else 2) and torch.equal(got[held], want[held])


@pytest.mark.parametrize("T,E,rows", [
    (6, 4, 16),          # unsorted
    (36, 10, 16),        # sorted
    (40, 9, 32),
    (40, 4, 64),
])
def test_wide_block_scales_equal_the_stages_within_rounding(T, E, rows):
    """MXFP4 activations whose block scales lie 2^20 apart along a row of the down GEMM (rows of w1 scaled by 2^-10, 1 and 2^10, 32 at a time;
    the gate_up GEMM's sums stay exact, so both paths have the same intermediate).  There n = K / 32 partial sums of a magnitude of at
    most S = sum |a2 * w2| are added in two orders: at most 2 n 2^-24 S between them, the routing weight and the bf16 rounding of the
    slot on top (half an ulp, 2^-9 of the value, on either side)."""
    import numpy as np
    from oracle import mxfp4
    from pyhip_amd import fused_moe
    H, I, k = 512, 2048, 2
    L = cases.make_layer("", T, seed=T, E=E, k=k, H=H, I=I, router="softmax")
    up = L.w1s.reshape(E, 2, I // 32, 32, H // 32)[:, 1]           # (a view: the up halves' scale bytes)
    up[:, 0::3] -= 10
    up[:, 2::3] += 10
    w1, w1s, w2, w2s = cases.device_weights(L)
    args = (L.hidden.cuda(), w1, w2, torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda())
    kw = dict(w1_scale=w1s, w2_scale=w2s, method="a4w4", block_size_M=rows, dtype=torch.float32)
    print("few pairs, wide scales", T, E, rows, flush=True)
    want, parts = fused_moe(*args, return_parts=True, **kw)
    _poison(T, k, E, H, I, "a4w4", rows)
    got = fused_moe(*args, **kw)
    a2_q, a2_s = parts["a2_q"].cpu().numpy(), cases.untranspose_act_scales(parts["a2_s"].cpu().numpy(), I)
    ids = parts["sorted_ids"].cpu().numpy().astype(np.int64)[:int(parts["num_valid_ids"][0])] & 0xFFFFFFFF
    bound = np.zeros((T, H))
    for p, (tok, slot) in enumerate(zip(ids & 0xFFFFFF, ids >> 24)):
        if tok < T and slot < k:
            e, a2 = L.topk_ids[tok, slot], mxfp4.dequantize_mxfp4(a2_q[p], a2_s[p])
            S = np.abs(mxfp4.dequantize_mxfp4(L.w2q[e], L.w2s[e])).astype(np.float64) @ np.abs(a2).astype(np.float64)
            bound[tok] += 2 * (I // 32) * 2.0 ** -24 * S * L.topk_w[tok, slot]
    bound += 2.0 ** -8 * parts["out3"].float().abs().sum(dim=1).cpu().numpy()
    diff = (got - want).abs().cpu().numpy()
    print("  differ:", (diff > 0).mean(), "largest share of the bound:", (diff / bound).max(), flush=True)
    assert np.isfinite(diff).all() and (diff <= bound).all(), (diff / bound).max()
    assert want.abs().mean() > 100 * bound.mean()                  # (the bound says something)


@pytest.mark.parametrize("T,k,E,H,I,method,rows", [
    (1, 8, 16, 512, 1536, "w4a16", 16),      # a token's slots of 12288 columns together: summed in the down GEMM
    (1, 8, 16, 512, 2048, "w4a16", 16),      # of more: by expert, and reduced
    (2, 5, 80, 512, 2560, "w4a16", 16),
    (64, 8, 128, 512, 512, "a4w4", 16),      # four rows per expert, but too many workgroups of one K-step
    (80, 2, 40, 512, 512, "a4w4", 16),       # sorted, four rows per expert, few workgroups
    (72, 2, 32, 2560, 512, "a4w4", 32),      # the same in 32 rows, an uneven share of K-steps
    (70, 1, 5, 5120, 512, "a4w4", 32),       # a handful of experts, twelve rows and more, a long K loop
])
def test_lines_of_the_few_token_kernels(T, k, E, H, I, method, rows):
    """on both sides of the lines by the length of the K loops: the bits of the stages one by one"""
    from pyhip_amd import fused_moe
    L = cases.make_layer("", T, seed=T, E=E, k=k, H=H, I=I, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    args = (L.hidden.cuda(), w1, w2, torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda())
    kw = dict(w1_scale=w1s, w2_scale=w2s, method=method, block_size_M=rows)
    print("few pairs, lines", T, k, E, H, I, method, rows, flush=True)
    want = fused_moe(*args, return_parts=True, **kw)[0]
    _poison(T, k, E, H, I, method, rows)
    assert torch.equal(fused_moe(*args, **kw), want)
