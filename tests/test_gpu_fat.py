"""GPU parity of the fat-expert path: per-expert grouped GEMM with the EXL3 weights decoded into LDS (fp16) and
multiplied on MFMA, fused output transforms / SwiGLU / down-input transform, and the prefill layer."""
import os

import numpy as np
import pytest

from helpers import OracleLayer, make_store, within_tolerance

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def test_fat_expert_matches_reference_golden(dev):
    """The two experts of the compiled reference's golden file, each fed 130 routes (a tile of 96 and one of 34),
    through the grouped GEMM: every route's row equals the reference's output."""
    import torch
    from mi355moe import moe
    g = np.load(os.path.join(GOLD, "expert_4096x2048.npz"), allow_pickle=False)
    H, I = int(g["H"]), int(g["I"])
    E = 256
    st = make_store(E, H, I, int(g["layer_seed"]), device=dev, exact=True)
    es = [int(g["e0"]), int(g["e1"])]
    for j, e in enumerate(es):
        st.w13_suh[e, 0].copy_(_t(g[f"suh_g{j}"], dev)); st.w13_svh[e, 0].copy_(_t(g[f"svh_g{j}"], dev))
        st.w13_suh[e, 1].copy_(_t(g[f"suh_u{j}"], dev)); st.w13_svh[e, 1].copy_(_t(g[f"svh_u{j}"], dev))
        st.w2_suh[e].copy_(_t(g[f"suh_d{j}"], dev)); st.w2_svh[e].copy_(_t(g[f"svh_d{j}"], dev))
    R = 130
    x = np.concatenate([np.repeat(g["x0"][None, :], R, 0), np.repeat(g["x1"][None, :], R, 0)]).astype(np.float16)
    ids = np.array([[es[0]]] * R + [[es[1]]] * R, np.int64)
    for lim in (10, 0):
        st.limit = float(lim)
        st._c = None
        print(f"fat golden limit {lim}", flush=True)
        Y = moe.grouped_gemm(st, _t(x, dev), _t(ids, dev), cap=0)
        torch.cuda.synchronize()
        Yg = Y.cpu().numpy()
        for j in (0, 1):
            ref = np.repeat(g[f"y{j}_lim{lim}"][None, :], R, 0)
            ok, m = within_tolerance(Yg[j * R:(j + 1) * R], ref)
            assert ok, (j, m)


@pytest.mark.parametrize("H,I,E,T,k", [(256, 128, 4, 200, 2), (512, 384, 6, 300, 3), (1024, 256, 3, 150, 2)])
def test_fat_small_shapes_vs_oracle(dev, H, I, E, T, k):
    import torch
    from mi355moe import moe
    seed = 777 + H + I
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(H * 3 + I)
    ids = np.stack([rng.choice(E, k, replace=False) for _ in range(T)]).astype(np.int64)
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"fat small H={H} I={I} E={E} T={T} k={k}", flush=True)
    out = moe.moe_prefill(st, _t(x16, dev), _t(ids, dev), _t(w, dev))
    torch.cuda.synchronize()
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    ok, m = within_tolerance(out.cpu().numpy(), ref)
    assert ok, m


def test_fat_tile_boundaries(dev):
    """Experts with 1, 128, 129, 192, 256 and 257 routes: tiles of up to 96 routes, full and with a remainder of one route or
    of one or two row groups of 32 (the larger tiles: test_tiles_of_sorted_experts and the large-layer test)."""
    import torch
    from mi355moe import moe
    H, I, seed = 256, 128, 8080
    counts = [1, 128, 129, 192, 256, 257]
    E = len(counts)
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(12)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int64)[:, None]
    T = ids.shape[0]
    w = np.ones((T, 1), np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"fat tile boundaries T={T}", flush=True)
    out = moe.moe_prefill(st, _t(x16, dev), _t(ids, dev), _t(w, dev))
    torch.cuda.synchronize()
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    for e in range(E):
        rows = ids[:, 0] == e
        ok, m = within_tolerance(out.cpu().numpy()[rows], ref[rows])
        assert ok, (counts[e], m)


def test_grouped_gemm_rows_of_fat_experts_only(dev):
    """Only routes of experts above cap get rows; masked ids (-1, >= E) and small experts are left untouched."""
    import torch
    from mi355moe import moe
    H, I, E, T, k = 512, 256, 6, 160, 2
    seed = 4321
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(8)
    ids = np.stack([rng.choice(E, k, replace=False) for _ in range(T)]).astype(np.int64)
    ids[ids == 5] = 4                                  # expert 4 busy, expert 5 idle
    ids[:, 1] = np.where(ids[:, 0] == 4, 2, ids[:, 1])  # no token picks 4 twice
    ids[::3, 1] = 1                                    # expert 1 busy too
    ids[np.arange(T) % 7 == 2, 0] = -1
    ids[np.arange(T) % 11 == 5, 1] = E + 3
    counts = np.bincount(ids[(ids >= 0) & (ids < E)], minlength=E)
    cap = int(np.sort(counts)[-3])                     # the two busiest experts are fat
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"grouped gemm cap={cap} counts={counts.tolist()}", flush=True)
    Y = moe.grouped_gemm(st, _t(x16, dev), _t(ids, dev), cap=cap)
    torch.cuda.synchronize()
    Yg = Y.cpu().numpy()
    flat = ids.reshape(-1)
    fat = (flat >= 0) & (flat < E) & (counts[np.clip(flat, 0, E - 1)] > cap)
    assert fat.sum() > 128 and (~fat).sum() > 0
    assert np.all(Yg[~fat] == 0.0)
    ref = OracleLayer(st, seed).per_route(x16.astype(np.float32), ids)
    ok, m = within_tolerance(Yg[fat], ref[fat])
    assert ok, m


def test_threshold_split_matches_oracle(dev):
    """moe_forward above the threshold, busy experts and experts with a few routes in one call of 240 routes (the decode
    path takes it whole), and the same routes divided by the threshold over both paths: mm_moe_decode leaves out the experts
    above max_rows, mm_moe_prefill with cap and accumulate adds them."""
    import torch
    from mi355moe import moe
    H, I, E, T, k = 512, 256, 8, 120, 2
    seed = 515
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(12)
    p = np.array([0.4, 0.3, 0.1, 0.08, 0.05, 0.04, 0.02, 0.01])
    ids = np.stack([rng.choice(E, k, replace=False, p=p) for _ in range(T)]).astype(np.int64)
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    counts = np.bincount(ids.reshape(-1), minlength=E)
    print(f"threshold split counts={counts.tolist()}", flush=True)
    assert (counts > 40).any() and ((counts > 0) & (counts <= 40)).any()
    out = moe.moe_forward(st, _t(x16, dev), _t(ids, dev), _t(w, dev), fat_threshold=40)
    few = moe.decode_routes(st, _t(x16, dev), _t(ids, dev), _t(w, dev), 40)
    split = moe.moe_prefill(st, _t(x16, dev), _t(ids, dev), _t(w, dev), cap=40, out=few.clone())
    torch.cuda.synchronize()
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    for got in (out, split):
        ok, m = within_tolerance(got.cpu().numpy(), ref)
        assert ok, m
    ok, m = within_tolerance(few.cpu().numpy(), OracleLayer(st, seed).forward(x16.astype(np.float32),
                                                                              np.where(counts[ids] > 40, -1, ids), w))
    assert ok, m


def test_prefill_full_shape_matches_decode_path(dev):
    """H 4096, I 2048, 384 routed + 1 shared expert, top-8 Zipf routing over 256 tokens: the prefill layer equals
    the decode path (every expert <= 256 routes) with fp16 weights, and the oracle on sampled tokens."""
    import torch
    from mi355moe import moe, workload
    H, I, E, T = 4096, 2048, 384, 256
    seed = 3100
    st = make_store(E + 1, H, I, seed, device=dev, exact=True)
    ids, w = workload.zipf_routing(T, 8, E, seed=3101)
    x16 = workload.activations(T, H, seed=3102).astype(np.float16)
    xd, idd, wd = _t(x16, dev), _t(ids, dev), _t(w, dev)
    print("prefill full shape T=256", flush=True)
    a = moe.moe_prefill(st, xd, idd, wd, shared_expert=E)
    b = moe.moe_forward(st, xd, idd, wd, shared_expert=E, fat_threshold=T)
    torch.cuda.synchronize()
    a, b = a.cpu().numpy(), b.cpu().numpy()
    ok, m = within_tolerance(a, b.astype(np.float64))
    print("prefill vs decode", m, flush=True)
    assert ok, m
    rows = [0, 97, 255]
    ids_ext = np.concatenate([ids, np.full((T, 1), E)], 1)
    w_ext = np.concatenate([w, np.ones((T, 1), np.float32)], 1)
    ref = OracleLayer(st, seed).forward(x16[rows].astype(np.float32), ids_ext[rows], w_ext[rows])
    ok, m = within_tolerance(a[rows], ref)
    assert ok, m


def test_prefill_16k_tokens_deterministic_and_sampled(dev):
    """The 16k-token prefill layer (16384 tokens, top-8 Zipf over 384 experts + shared): two runs are bit-equal,
    accumulate adds onto out, and sampled tokens match the oracle."""
    import torch
    from mi355moe import moe, workload
    H, I, E, T = 4096, 2048, 384, 16384
    seed = 3200
    st = make_store(E + 1, H, I, seed, device=dev, exact=True)
    ids, w = workload.zipf_routing(T, 8, E, seed=3201)
    x16 = workload.activations(T, H, seed=3202).astype(np.float16)
    xd, idd, wd = _t(x16, dev), _t(ids, dev), _t(w, dev)
    print("prefill 16k tokens", flush=True)
    a = moe.moe_prefill(st, xd, idd, wd, shared_expert=E)
    b = moe.moe_prefill(st, xd, idd, wd, shared_expert=E)
    c = moe.moe_prefill(st, xd, idd, wd, shared_expert=E, out=a.clone())
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    # accumulate: out starts from a and adds the same routes in the same order
    assert torch.allclose(c, a + a, rtol=1e-5, atol=1e-5 * float(a.abs().max()))
    rows = [0, 8191, 16383]
    ids_ext = np.concatenate([ids, np.full((T, 1), E)], 1)
    w_ext = np.concatenate([w, np.ones((T, 1), np.float32)], 1)
    ref = OracleLayer(st, seed).forward(x16[rows].astype(np.float32), ids_ext[rows], w_ext[rows])
    ok, m = within_tolerance(a.cpu().numpy()[rows], ref)
    print("16k sampled", m, flush=True)
    assert ok, m


@pytest.mark.parametrize("T,k,E,cap", [(600, 4, 40, 32), (90, 6, 24, 20)])
def test_fused_moe_device_split_vs_oracle(dev, T, k, E, cap):
    """mm_fused_moe on the grouped GEMM (2,400 routes) and on the decode path (540), experts above and below cap, which
    chooses nothing: two runs are bit-equal and match the oracle."""
    import torch
    from mi355moe import moe
    H, I = 512, 256
    seed = 7700 + T
    st = make_store(E, H, I, seed, device=dev)
    rng = np.random.default_rng(T)
    p = np.concatenate([np.full(E // 4, 3.0), np.ones(E - E // 4)])
    p /= p.sum()
    ids = np.stack([rng.choice(E, k, replace=False, p=p) for _ in range(T)]).astype(np.int64)
    ids[::11, 1] = -1
    counts = np.bincount(ids[ids >= 0], minlength=E)
    assert (counts > cap).any() and ((counts > 0) & (counts <= cap)).any()
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"fused device split T={T} k={k} counts={counts.tolist()}", flush=True)
    out = moe.fused_moe(st, _t(x16, dev), _t(ids, dev), _t(w, dev), cap)
    again = moe.fused_moe(st, _t(x16, dev), _t(ids, dev), _t(w, dev), cap)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    ok, m = within_tolerance(out.cpu().numpy(), ref)
    assert ok, m


@pytest.mark.parametrize("exact", [True, False])
def test_row_group_tiles_at_their_edges(dev, exact):
    """Experts whose routes end on either side of the row groups of 32, of the tiles of 96 and of 192, through the grouped
    GEMM (fp16-rounded weights) and through a fused call of more than 1,024 routes (the layer's evaluation), down GEMM
    of four steps (two per half of K)."""
    import torch
    from mi355moe import moe
    H, I, seed = 512, 128, 8181
    counts = [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 256, 289]
    E = len(counts)
    st = make_store(E, H, I, seed, device=dev, exact=exact)
    rng = np.random.default_rng(13)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int64)[:, None]
    T = ids.shape[0]
    w = np.ones((T, 1), np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"row group tiles T={T} exact={exact}", flush=True)
    assert T > 1024
    Y = moe.grouped_gemm(st, _t(x16, dev), _t(ids, dev), cap=0)
    out = moe.fused_moe(st, _t(x16, dev), _t(ids, dev), _t(w, dev), 32)
    torch.cuda.synchronize()
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    for e in range(E):
        rows = ids[:, 0] == e
        for name, got in (("grouped", Y), ("fused", out)):
            ok, m = within_tolerance(got.cpu().numpy()[rows], ref[rows])
            assert ok, (name, counts[e], m)


@pytest.mark.parametrize("exact", [True, False])
def test_full_tiles_of_a_large_call(dev, exact):
    """Enough 256-route tiles to take their own kernels (at least three rounds of 256 workgroups of them), with remainders
    of one route, of one and of two row groups, and partial tiles of 193 and 255 routes: sampled rows of every expert. In a
    layer without MM_LAYER_EXACT the 256-route tiles round the weights and write no input sums, the others need them."""
    import torch
    from mi355moe import moe
    H, I, seed = 256, 2048, 8282
    counts = [193, 255, 256, 257, 290, 330] * 9
    E = len(counts)
    assert sum(c // 256 + (c % 256 >= 193) for c in counts) * (I // 128) >= 3 * 256
    st = make_store(E, H, I, seed, device=dev, exact=exact)
    rng = np.random.default_rng(14)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int64)[:, None]
    T = ids.shape[0]
    w = np.ones((T, 1), np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    print(f"full tiles T={T} exact={exact}", flush=True)
    out = moe.fused_moe(st, _t(x16, dev), _t(ids, dev), _t(w, dev), 32)
    torch.cuda.synchronize()
    rows = np.concatenate([np.flatnonzero(ids[:, 0] == e)[[0, 100, 192, -1]] for e in range(E)])
    ref = OracleLayer(st, seed).forward(x16[rows].astype(np.float32), ids[rows], w[rows])
    ok, m = within_tolerance(out.cpu().numpy()[rows], ref)
    assert ok, m


@pytest.mark.parametrize("E,H,I,T,k,hot,path", [
    (8, 4096, 2048, 192, 2, 8, "decode"), (8, 4096, 2048, 193, 2, 8, "gemm"), (20, 4096, 2048, 52, 8, 20, "decode"),
    (20, 4096, 2048, 53, 8, 20, "gemm"), (8, 256, 128, 1024, 1, 8, "decode"), (8, 256, 128, 1025, 1, 8, "gemm"),
    (1024, 1024, 1024, 1025, 1, 90, "decode"), (1024, 1024, 1024, 1025, 1, 12, "gemm"),
    (1024, 1024, 1024, 540, 2, 110, "decode"), (1024, 1024, 1024, 540, 2, 8, "gemm"), (1024, 1024, 1024, 1195, 6, 12, "gemm")])
def test_fused_call_on_either_side_of_its_path_rule(dev, E, H, I, T, k, hot, path):
    """Fused calls at the last routes of the decode path and the first of the grouped GEMM (384 routes, or 10 per expert and
    220 at H 4096, I 2048, more in smaller layers), and above 1,024 routes of large layers on either side of the choice made
    on the device (up to 7 routes per expert; by records of 16 and tiles of 96 routes): nothing is written past the workspace
    asked for, stale workspace is not read, the decode path's calls equal it bit for bit whatever the threshold, and every
    call matches the oracle."""
    import torch
    from mi355moe import _lib, moe
    seed = 9300 + E
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(T)
    ids = np.stack([rng.choice(hot, k, replace=False) for _ in range(T)]).astype(np.int64)
    ids[::13, k - 1] = -1
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    n = T * k
    counts = np.bincount(ids[ids >= 0], minlength=E)
    if n <= 1024:
        decode = n <= max(384, 10 * E + 220 * 4096 * 2048 // (H * I))
    else:
        chosen = n <= min(9 * E, max(7 * E, 1280)) and E * H * I >= 1 << 30
        decode = chosen and 800 * np.sum(-(-counts // 16)) + 8 * n <= 900 * np.sum(-(-counts // 96)) + 10400
    assert decode == (path == "decode")
    print(f"fused call E={E} T={T} k={k} hot={hot} ({path})", flush=True)
    xd, idd, wd = _t(x16, dev), _t(ids, dev), _t(w, dev)
    wsb = _lib.load().mm_fused_moe_workspace(T, k, E, H, I, 32)
    ws = torch.full((wsb + 4096,), 0xff, dtype=torch.uint8, device=dev)     # NaNs before, guard bytes behind
    out = torch.empty((T, H), dtype=torch.float32, device=dev)
    _lib.call("mm_fused_moe", st.mm_layer(), xd.data_ptr(), _lib.DTYPE_F16, T, k, idd.data_ptr(), wd.data_ptr(), 32,
              out.data_ptr(), ws.data_ptr(), wsb, _lib.stream_ptr())
    again = moe.fused_moe(st, xd, idd, wd, 1)
    routed = moe.decode_routes(st, xd, idd, wd, n)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and (ws[wsb:] == 0xff).all().item()
    assert torch.equal(out, routed) == (path == "decode")
    rows = np.arange(0, T, max(1, T // 40 if H == 4096 else T // 200))
    ref = OracleLayer(st, seed).forward(x16[rows].astype(np.float32), ids[rows], w[rows])
    ok, m = within_tolerance(out.cpu().numpy()[rows], ref)
    assert ok, m


def test_fused_call_chosen_on_the_device_in_a_graph(dev):
    """A captured call of more than 1,024 routes in the range where the device chooses the path: replays with routes that
    take the decode path, the grouped GEMM, nothing (every id masked: zeros) and the decode path again equal the eager calls
    bit for bit."""
    import torch
    from mi355moe import moe
    H, I, E, T = 1024, 1024, 1024, 1100
    st = make_store(E, H, I, 9400, device=dev)
    rng = np.random.default_rng(3)
    x = _t(rng.normal(0, 1, (T, H)).astype(np.float16), dev)
    w = _t(rng.uniform(0.1, 1.0, (T, 1)).astype(np.float32), dev)
    wide, few, none = (_t(v.astype(np.int64), dev) for v in (rng.integers(0, E, (T, 1)), rng.integers(0, 6, (T, 1)),
                                                             np.full((T, 1), -1)))
    print("fused call chosen in a graph", flush=True)
    eager = [moe.fused_moe(st, x, i, w, 32) for i in (wide, few, none)]
    torch.cuda.synchronize()
    assert torch.equal(eager[0], moe.decode_routes(st, x, wide, w, T))
    assert not torch.equal(eager[1], moe.decode_routes(st, x, few, w, T)) and torch.count_nonzero(eager[2]).item() == 0
    ids = wide.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = moe.fused_moe(st, x, ids, w, 32)
    for step, (i, want) in enumerate(zip((wide, few, none, wide), (eager[0], eager[1], eager[2], eager[0]))):
        ids.copy_(i)
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {step}"


def test_tiles_of_sorted_experts(dev):
    """apply_exl3_batched_fat takes 256-route tiles by the expert's own routes, from 768 on: 767 to 1,025 routes, every row
    against the oracle, and an expert computed alone has the bits it has among the others."""
    import torch
    from mi355moe import exl3, moe
    H, I, seed = 512, 256, 8484
    counts = [767, 768, 769, 960, 961, 1025]
    E = len(counts)
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(17)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int64)[:, None]
    T = ids.shape[0]
    w = np.ones((T, 1), np.float32)
    x16 = rng.normal(0, 1, (T, H)).astype(np.float16)
    xd = _t(x16, dev)
    r = moe.permute(_t(ids, dev), _t(w, dev), 1, E)
    tok, wts = r["token_sorted"].long(), r["weight_sorted"].half()
    print(f"sorted experts T={T}", flush=True)

    def run(skip):
        o = torch.zeros((T, H), dtype=torch.float32, device=dev)
        return exl3.apply_exl3_batched_fat(xd, tok, wts, counts, None, 10.0, 0, o, skip=skip, layer=st)

    out = run(None)
    alone = sum(run(set(range(E)) - {e}) for e in range(E))
    torch.cuda.synchronize()
    assert torch.equal(out, alone)
    ref = OracleLayer(st, seed).forward(x16.astype(np.float32), ids, w)
    for e in range(E):
        rows = ids[:, 0] == e
        ok, m = within_tolerance(out.cpu().numpy()[rows], ref[rows])
        assert ok, (counts[e], m)


@pytest.mark.parametrize("more", [[], [1, 17, 32, 33, 64, 95, 96] * 2], ids=["folded", "all_sizes"])
def test_tiles_of_a_large_rounding_layer(dev, more):
    """Layers of at least 80,000 routes and 200 per expert: remainders of 97 to 128 routes in 128-route tiles, from 129 on in
    256-route tiles (with remainders of 1, 96, 97 and 128 after full ones), and the shorter ones in 128-route tiles too where
    the layer has few of them (an 18th of a round of workgroups here), else in tiles of their own. mm_grouped_gemm, mm_moe_prefill
    and apply_exl3_batched_fat, the last in one call and in batches, give every row the same bits; sampled rows of every
    expert against the oracle."""
    import torch
    from mi355moe import exl3, moe
    H, I, seed = 256, 4096, 8585
    counts = [97, 112, 113, 128, 129, 176, 255, 256, 257, 352, 353, 384, 31, 32, 96] + more
    shorter = sum(0 < c % 256 <= 96 for c in counts)
    counts.append(80256 - sum(counts) - (80256 - sum(counts)) % 256)
    assert (shorter <= 12) == (not more) and 80000 <= sum(counts)   # half of 24 tiles = 768 workgroups of I / 128
    E = len(counts)
    st = make_store(E, H, I, seed, device=dev, exact=True)
    rng = np.random.default_rng(18)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int64)[:, None]
    T = ids.shape[0]
    xd = torch.randn((T, H), generator=torch.Generator(device=dev).manual_seed(18), device=dev).half()
    idd, w = _t(ids, dev), torch.ones((T, 1), device=dev)
    r = moe.permute(idd, w, 1, E)
    tok, wts = r["token_sorted"].long(), r["weight_sorted"].half()
    print(f"large rounding layer T={T} experts={E}", flush=True)

    def run(skip):
        o = torch.zeros((T, H), dtype=torch.float32, device=dev)
        return exl3.apply_exl3_batched_fat(xd, tok, wts, counts, None, 10.0, 0, o, skip=skip, layer=st)

    Y = moe.grouped_gemm(st, xd, idd, cap=0)
    out = moe.moe_prefill(st, xd, idd, w)
    whole = run(None)
    parts = sum(run(set(range(E)) - set(range(b, E, 4))) for b in range(4))
    torch.cuda.synchronize()
    assert torch.equal(Y.half().float(), out) and torch.equal(whole, out) and torch.equal(parts, out)
    at = [np.flatnonzero(ids[:, 0] == e) for e in range(E)]
    rows = np.concatenate([q[np.unique(np.minimum([0, len(q) // 2, 96, 128, len(q) - 1], len(q) - 1))] for q in at])
    ref = OracleLayer(st, seed).forward(xd[_t(rows, dev)].float().cpu().numpy(), ids[rows], np.ones((len(rows), 1), np.float32))
    ok, m = within_tolerance(Y.cpu().numpy()[rows], ref)
    assert ok, m


def test_full_tiles_match_reference_golden(dev):
    """The compiled reference's golden experts with 800 routes each (three 256-route tiles and a row group) through
    apply_exl3_batched_fat: every route's row equals the reference's output."""
    import torch
    from mi355moe import exl3
    g = np.load(os.path.join(GOLD, "expert_4096x2048.npz"), allow_pickle=False)
    H, I, R = int(g["H"]), int(g["I"]), 800
    st = make_store(256, H, I, int(g["layer_seed"]), device=dev, exact=True)
    es = [int(g["e0"]), int(g["e1"])]
    for j, e in enumerate(es):
        st.w13_suh[e, 0].copy_(_t(g[f"suh_g{j}"], dev)); st.w13_svh[e, 0].copy_(_t(g[f"svh_g{j}"], dev))
        st.w13_suh[e, 1].copy_(_t(g[f"suh_u{j}"], dev)); st.w13_svh[e, 1].copy_(_t(g[f"svh_u{j}"], dev))
        st.w2_suh[e].copy_(_t(g[f"suh_d{j}"], dev)); st.w2_svh[e].copy_(_t(g[f"svh_d{j}"], dev))
    x = _t(np.stack([g["x0"], g["x1"]]).repeat(R, 0).astype(np.float16), dev)
    order = sorted((0, 1), key=lambda j: es[j])
    tok = torch.cat([torch.arange(j * R, (j + 1) * R, device=dev) for j in order])
    counts = [R if e in es else 0 for e in range(256)]
    out = torch.zeros((2 * R, H), dtype=torch.float32, device=dev)
    print("golden experts in full tiles", flush=True)
    exl3.apply_exl3_batched_fat(x, tok, torch.ones(2 * R, device=dev).half(), counts, None, 10.0, 0, out, layer=st)
    torch.cuda.synchronize()
    for j in (0, 1):
        ok, m = within_tolerance(out.cpu().numpy()[j * R:(j + 1) * R], np.repeat(g[f"y{j}_lim10"][None, :], R, 0))
        assert ok, (j, m)
