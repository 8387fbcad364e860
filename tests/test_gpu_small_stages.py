"""The small stages around the GEMMs at the sizes where their split over waves has edges."""
import numpy as np
import pytest
import torch

from pyhip_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (3, 2, 504), (2, 8, 512), (5, 9, 520), (7, 4, 1032), (2, 33, 2880), (4001, 8, 256)])
@pytest.mark.parametrize("mode", ["plain", "ids", "mask", "local"])
@pytest.mark.parametrize("f32", [False, True])
def test_topk_reduce_edges(T, k, H, mode, f32):
    """Rows that are no whole number of 64-lane pieces, slots past one group of eight, dropped slots that hold NaN; against
    numpy's sums in slot order, which the kernel's single-precision additions must equal exactly."""
    g = torch.Generator().manual_seed(T * 100 + k)
    E = 16
    x = torch.randn(T, k, H, generator=g).to(torch.bfloat16)
    ids = torch.randint(0 if mode == "plain" else -1, E if mode == "plain" else E + 1, (T, k), generator=g, dtype=torch.int32)
    mask = (torch.arange(E) % 3 != 0).to(torch.int32) if mode == "mask" else None
    local = torch.tensor([T // 2], dtype=torch.int32) if mode == "local" else None
    keep = (ids >= 0) & (ids < E)
    if mask is not None:
        keep &= mask[ids.clamp(0, E - 1).long()] != 0
    if local is not None:
        keep &= (torch.arange(T) < T // 2)[:, None]
    x[~keep] = float("nan")
    ref = np.zeros((T, H), np.float32)
    xf = x.float().numpy()
    for s in range(k):
        ref += np.where(keep[:, s, None].numpy(), xf[:, s], np.float32(0))
    lib = _lib.load()
    P = _lib.dptr
    xd, idd = x.cuda(), ids.cuda()
    md, ld = (None if v is None else v.cuda() for v in (mask, local))
    out = torch.full((T, H), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    print("topk_reduce", T, k, H, mode, f32, flush=True)
    if mode == "plain":
        _lib.check(lib.pyhip_moe_topk_reduce(P(xd), P(out), T, k, H, int(f32), None, _lib.current_stream()))
    else:
        _lib.check(lib.pyhip_moe_topk_reduce_routed(P(xd), P(out), T, k, H, int(f32), P(idd), E, P(md), P(ld),
                                                    _lib.current_stream()))
    want = torch.from_numpy(ref)
    assert torch.equal(out.cpu(), want if f32 else want.to(torch.bfloat16))


@pytest.mark.parametrize("T,k", [(1, 1), (63, 1), (64, 1), (65, 1), (31, 8), (129, 8), (255, 4), (1025, 1), (256, 8)])
@pytest.mark.parametrize("E,masked", [(1, False), (8, False), (63, True), (256, True), (1040, False)])
def test_single_workgroup_sort_edges(T, k, E, masked):
    """One wave with pairs, two, all sixteen with one or two groups each; fewer experts than lanes, more than threads:
    the positions an expert-by-expert walk on the CPU gives."""
    from pyhip_amd.moe_sorting import moe_sorting
    rng = np.random.default_rng(T * 1000 + E)
    ids = rng.integers(0, E, (T, k)).astype(np.int32)
    w = rng.random((T, k), dtype=np.float32)
    mask = (rng.random(E) < 0.7).astype(np.int32) if masked else None
    bm = 32
    so, sw, se = [], [], []
    local = 0
    for e in range(E):
        if mask is not None and not mask[e]:
            continue
        t, s = np.nonzero(ids == e)
        fill = -len(t) % bm
        so += [(int(b) << 24) | int(a) for a, b in zip(t, s)] + [(k << 24) | T] * fill
        sw += list(w[t, s]) + [0.0] * fill
        se += [local] * ((len(t) + fill) // bm)
        local += 1
    print("sort", T, k, E, masked, flush=True)
    got = moe_sorting(torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(), E, 256, torch.bfloat16, bm,
                      None if mask is None else torch.from_numpy(mask).cuda(), alloc_moe_out=False)
    n = int(got[3][0])
    assert n == len(so) and int(got[3][1]) == T
    assert (got[0].cpu().numpy().view(np.uint32)[:n] == np.array(so, np.uint32)).all()
    assert (got[1].cpu().numpy()[:n] == np.array(sw, np.float32)).all()
    assert (got[2].cpu().numpy().view(np.uint32)[:n // bm] == np.array(se, np.uint32)).all()


@pytest.mark.parametrize("E", [64, 128, 256, 512])
@pytest.mark.parametrize("grouped", [False, True])
def test_router_ties_and_missing_scores(E, grouped):
    """Equal scores go to the lower expert, minus infinity ranks last: the picks of a stable descending sort."""
    from pyhip_amd.routing import fused_topk, grouped_topk
    g = torch.Generator().manual_seed(E)
    T, k = 37, 8
    x = torch.randint(-3, 4, (T, E), generator=g).float()          # seven distinct scores: ties everywhere
    x[0] = 0.0
    x[1, :E - 1] = float("-inf")
    x[2, ::2] = float("-inf")
    x[3] = torch.arange(E).float().flip(0) / 64
    s = torch.sigmoid(x) if grouped else torch.softmax(x, dim=-1)
    if grouped:
        best = s.view(T, 8, -1).topk(2, dim=-1).values.sum(-1)
        groups = torch.sort(best, dim=-1, descending=True, stable=True).indices[:, :4]
        on = torch.zeros(T, 8, dtype=torch.bool).scatter_(1, groups, True)
        s = s.masked_fill(~on.repeat_interleave(E // 8, dim=1), float("-inf"))
    want = torch.sort(s, dim=-1, descending=True, stable=True).indices[:, :k]
    print("router", E, grouped, flush=True)
    dev = x.cuda()
    hidden = torch.zeros(T, 64, dtype=torch.bfloat16, device="cuda")
    got = grouped_topk(dev, k, True, 8, 4) if grouped else fused_topk(hidden, dev, k, True)
    assert torch.equal(got[1].cpu().long(), want)


@pytest.mark.parametrize("T", [5, 65, 600])
@pytest.mark.parametrize("form", ["contiguous", "row_stride", "odd_stride", "misaligned", "expanded", "transposed"])
def test_true_width_activations(T, form):
    """A padded layer called with activations at the true width, in every form they may come in, against the same
    values widened by the caller: the same bits, and the widened shape's result cut to the true width."""
    import cases
    from pyhip_amd import fused_moe
    L = cases.make_layer("gptoss_s", T, seed=5, bias=True)
    w1, w1s, w2, w2s, b1, b2, hp, ip = cases.padded_device_weights(L)
    tw, ti = torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda()
    x, H = L.hidden.cuda(), L.H
    if form == "row_stride":
        x = torch.nn.functional.pad(x, (0, 8), value=float("nan"))[:, :H]
    elif form == "odd_stride":
        x = torch.nn.functional.pad(x, (0, 3), value=float("nan"))[:, :H]
    elif form == "misaligned":
        buf = torch.empty(T * H + 1, dtype=x.dtype, device="cuda")
        buf[1:] = x.flatten()
        x = buf[1:].view(T, H)
    elif form == "expanded":
        x = x[:1].expand(T, H)
    elif form == "transposed":
        x = x.t().contiguous().t()
    kw = dict(w1_scale=w1s, w2_scale=w2s, bias1=b1, bias2=b2, hidden_pad=hp, intermediate_pad=ip)
    for method in ("auto", "a4w4", "w4a16"):
        print("true width", T, form, method, flush=True)
        got = fused_moe(x, w1, w2, tw, ti, method=method, **kw)
        wide = fused_moe(torch.nn.functional.pad(x, (0, hp)), w1, w2, tw, ti, method=method, **kw)
        assert got.shape == (T, H) and torch.equal(got, wide[:, :H])


@pytest.mark.parametrize("T", [5, 65, 600])
@pytest.mark.parametrize("option", ["mask", "many_experts", "local", "f32"])
def test_true_width_activations_with_options(T, option):
    """True-width rows of a padded layer under an expert mask (also over so many experts that the sort needs more than
    64 KB of LDS), a local token count and fp32 output: the bits of the same call with the rows widened by the caller."""
    import cases
    from pyhip_amd import fused_moe
    L = cases.make_layer("gptoss_s", T, seed=6, bias=True)
    w1, w1s, w2, w2s, b1, b2, hp, ip = cases.padded_device_weights(L)
    tw, ti = torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda()
    x = L.hidden.cuda()
    kw = dict(w1_scale=w1s, w2_scale=w2s, bias1=b1, bias2=b2, hidden_pad=hp, intermediate_pad=ip, method="a4w4")
    if option in ("mask", "many_experts"):
        # this rank's 16 experts among 48 or 1040: every third or sixty-fifth id
        step = 3 if option == "mask" else 65
        mask = torch.zeros(L.E * step, dtype=torch.int32)
        mask[::step] = 1
        kw["expert_mask"] = mask.cuda()
        ti = ti * step
        ti[:, 1] += 1                                  # a slot of experts that live elsewhere
    elif option == "local":
        kw["num_local_tokens"] = torch.tensor([T * 2 // 3], dtype=torch.int32, device="cuda")
        x = x.clone()
        x[T * 2 // 3:] = float("nan")                  # rows past the count are not looked at
    else:
        kw["dtype"] = torch.float32
    print("true width", T, option, flush=True)
    got = fused_moe(x, w1, w2, tw, ti, **kw)
    wide = fused_moe(torch.nn.functional.pad(x, (0, hp)), w1, w2, tw, ti, **kw)
    assert got.dtype == (torch.float32 if option == "f32" else torch.bfloat16) and torch.isfinite(got.float()).all()
    assert got.shape == (T, L.H) and torch.equal(got, wide[:, :L.H]) and got.float().abs().sum() > 0
