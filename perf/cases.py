"""What a user of this library has it do, as timed and checked cases: MoE layers of a decode step, the fused-MoE call of
batches and prefill chunks, one staged batch of busy experts, and the router, all on synthetic EXL3 experts.

A case names the entry point (`kind`), the expert shape, the routing and the number of tokens:

  layers   the MoE layers of one decode step (moe.DecodeRunner.layer), each on its own hidden states, routed experts
           plus the shared one
  call     the fused-MoE call of one layer: exl3.apply_exl3_fused_moe (routed experts), or moe.moe_forward when the
           shared expert takes part
  sorted   exl3.apply_exl3_batched_fat: the busy experts of one staging batch out of a prefill chunk
  router   mm_router_topk: logits, top-k and softmax weights

Expert shapes are the ones the library is built for: H 4096 / I 2048, 384 experts, top-8, and H 5120 / I 2304, 384
experts, top-6. Routing is Zipf(1.1) over a random ranking (decode) or 64 hot experts taking 60 % of the routes
(prefill chunks).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "dsv41-flash-offload_amd"))

from mi355moe import _lib, exl3, moe  # noqa: E402
from mi355moe.store import ExpertStore  # noqa: E402

E = 384
SHAPES = {"4096x2048": (4096, 2048, 8), "5120x2304": (5120, 2304, 6)}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
MOST_TOKENS = {"4096x2048": 16384, "5120x2304": 15360}      # the largest chunk (fewer tokens at the larger experts)
SHARED_MOST = 2048                                           # tokens of a drawn call with the shared expert


def _layers(name, tokens, shape="4096x2048", layers=6, dtype="f32", rescale=True, rounded=False, limit=10.0):
    return {"name": name, "kind": "layers", "tokens": tokens, "shape": shape, "layers": layers, "dtype": dtype,
            "rescale": rescale, "rounded": rounded, "limit": limit, "routing": "zipf"}


def _call(name, tokens, shape="4096x2048", dtype="bf16", routing="skewed", shared=False, rounded=False, limit=10.0):
    return {"name": name, "kind": "call", "tokens": tokens, "shape": shape, "dtype": dtype, "routing": routing,
            "shared": shared, "rounded": rounded, "limit": limit}


def listed():
    return [
        # one request decoding: the smallest call, six layers of the model in turn so that no layer's experts are
        # still in a cache when it comes round again
        _layers("decode 1 token", 1),
        # the batch the decode benchmark is quoted on
        _layers("decode 4 tokens", 4),
        # a speculative step of two requests with three tokens each on the larger experts, fp16-rounded weights
        _layers("decode 6 tokens 5120", 6, shape="5120x2304", layers=4, dtype="f16", rescale=False, rounded=True),
        # two dozen requests decoding together, with the shared expert
        _call("batch 24", 24, dtype="f16", routing="zipf", shared=True),
        # a hundred requests decoding together: a few busy experts, many with one or two rows
        _call("batch 100", 100, routing="zipf"),
        # a short prompt
        _call("prefill 512", 512, routing="zipf"),
        # prompts of odd length packed into one step: busy experts and experts with a few rows
        _call("prefill 1500", 1500, shared=True),
        # the usual prefill chunks of a server
        _call("prefill 4096", 4096),
        _call("prefill 8000 5120", 8000, shape="5120x2304"),
        # the largest chunk
        _call("prefill 16384", 16384),
        # one staging batch of 16 experts out of an 8,192-token chunk (experts that live in host memory)
        {"name": "staged batch", "kind": "sorted", "tokens": 8192, "shape": "4096x2048", "dtype": "f16",
         "routing": "skewed", "experts": 16, "cap": 0, "limit": 10.0},
        # the router of a mixed step
        {"name": "router 700", "kind": "router", "tokens": 700, "shape": "4096x2048"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["layers", "call", "sorted", "router"], [0.25, 0.5, 0.1, 0.15])[0]
    shape = rng.choice(["4096x2048", "4096x2048", "5120x2304"])
    if kind == "layers":
        rescale = rng.random() < 0.5
        return {"kind": kind, "tokens": _log_int(rng, 1, 32), "shape": shape, "layers": rng.randint(3, 6),
                "dtype": "f32" if rescale else rng.choice(["f16", "bf16"]), "rescale": rescale,
                "rounded": rng.random() < 0.25, "limit": rng.choice([10.0, 10.0, 0.0]), "routing": "zipf"}
    if kind == "call":
        shared = rng.random() < 0.3
        most = SHARED_MOST if shared else MOST_TOKENS[shape]
        return {"kind": kind, "tokens": _log_int(rng, 1, most), "shape": shape, "dtype": rng.choice(["f16", "bf16", "bf16"]),
                "routing": rng.choice(["zipf", "skewed"]), "shared": shared, "rounded": rng.random() < 0.2,
                "limit": rng.choice([10.0, 10.0, 0.0])}
    if kind == "sorted":
        return {"kind": kind, "tokens": _log_int(rng, 256, 8192), "shape": shape, "dtype": rng.choice(["f16", "bf16"]),
                "routing": rng.choice(["zipf", "skewed"]), "experts": rng.choice([8, 16, 24]), "cap": rng.choice([0, 32]),
                "limit": rng.choice([10.0, 0.0])}
    return {"kind": kind, "tokens": _log_int(rng, 1, 16384), "shape": shape}


# ------------------------------------------------------------------------------------------------- inputs

def _gen(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _routing(case, g, device):
    """ids int64 [T, k] of k distinct experts per token and softmax weights fp32 [T, k]."""
    T, k = case["tokens"], SHAPES[case["shape"]][2]
    if case["routing"] == "zipf":
        p = torch.arange(1, E + 1, dtype=torch.float64) ** -1.1
    else:
        p = torch.full((E,), 0.4 / (E - 64), dtype=torch.float64)
        p[:64] = 0.6 / 64
    perm = torch.randperm(E, generator=g, device=device)
    u = torch.rand((T, E), generator=g, device=device).clamp_(1e-7, 1 - 1e-7)
    keys = torch.log(p / p.sum()).float().to(device) - torch.log(-torch.log(u))
    ids = perm[torch.topk(keys, k, dim=1).indices]
    w = torch.softmax(torch.randn((T, k), generator=g, device=device), 1)
    return ids.contiguous(), w.contiguous()


def _store(case, n, g):
    """One layer's experts in HBM: random trellis words (every word is a valid code), +-1 input scales and half-normal
    output scales, as the synthetic checkpoints of the benchmark have."""
    H, I, _ = SHAPES[case["shape"]]
    st = ExpertStore(n, H, I, device="cuda", limit=case["limit"], exact=bool(case.get("rounded", False)))
    for t in (st.w13_trellis, st.w2_trellis):
        t.view(torch.int32).random_(-2 ** 31, 2 ** 31, generator=g)
    for t in (st.w13_suh, st.w2_suh):
        t.copy_(torch.randint(0, 2, t.shape, generator=g, device="cuda") * 2 - 1)
    for t in (st.w13_svh, st.w2_svh):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda").abs_() * 0.02)
    return st


def _hidden(case, g):
    """Hidden states N(0, 1), bf16-valued as a bf16 model hands them over; fp32 ones (the sum of a previous layer)
    keep all their bits and an RMS away from 1."""
    T, H = case["tokens"], SHAPES[case["shape"]][0]
    x = torch.randn((T, H), generator=g, device="cuda")
    return x * 0.3 if case["dtype"] == "f32" else x.bfloat16().to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = _gen(seed, "cuda")
    H, I, k = SHAPES[case["shape"]]
    T = case["tokens"]
    if case["kind"] == "router":
        return {"case": case, "x": torch.randn((T, H), generator=g, device="cuda").bfloat16(),
                "gate": torch.randn((E, H), generator=g, device="cuda") * 0.02,
                "logits": torch.empty((T, E), device="cuda"), "ids": torch.empty((T, k), dtype=torch.long, device="cuda"),
                "w": torch.empty((T, k), device="cuda")}
    if case["kind"] == "layers":
        r = moe.DecodeRunner(E, H, I, T, k)
        s = {"case": case, "runner": r, "stores": [], "x": [], "ids": [], "w": [], "out": []}
        for _ in range(case["layers"]):
            ids, w = _routing(case, g, "cuda")
            r.set_routes(ids, w)                      # the routed experts; the runner's last column is the shared one
            s["ids"].append(r.ids.clone())
            s["w"].append(r.w.clone())
            s["stores"].append(_store(case, E + 1, g))
            s["x"].append(_hidden(case, g))
            s["out"].append(torch.empty((T, H), device="cuda"))
        return s
    ids, w = _routing(case, g, "cuda")
    n = E + 1 if case.get("shared") else E
    s = {"case": case, "store": _store(case, n, g), "x": _hidden(case, g), "ids": ids, "w": w}
    if case["kind"] == "sorted":
        routes = moe.permute(ids, w, k, E)
        counts = routes["counts"][:E].cpu().numpy()
        s["token_sorted"] = routes["token_sorted"].long()
        s["weight_sorted"] = routes["weight_sorted"].half()
        s["counts"] = counts
        s["batch"] = sorted(np.random.default_rng(int(seed)).choice(E, case["experts"], replace=False).tolist())
        s["skip"] = set(range(E)) - set(s["batch"])
    return s


def run(state):
    case = state["case"]
    if case["kind"] == "layers":
        r = state["runner"]
        for st, x, ids, w, out in zip(state["stores"], state["x"], state["ids"], state["w"], state["out"]):
            r.layer(st, x=x, ids=ids, w=w, out=out, rescale=case["rescale"])
        return list(state["out"])
    if case["kind"] == "router":
        H, _, k = SHAPES[case["shape"]]
        _lib.call("mm_router_topk", state["x"].data_ptr(), case["tokens"], H, state["gate"].data_ptr(), E, k,
                  state["logits"].data_ptr(), state["ids"].data_ptr(), state["w"].data_ptr(), _lib.stream_ptr())
        return {"logits": state["logits"], "ids": state["ids"], "w": state["w"]}
    if case["kind"] == "sorted":
        out = torch.zeros(state["x"].shape, device="cuda")
        return exl3.apply_exl3_batched_fat(state["x"], state["token_sorted"], state["weight_sorted"], state["counts"],
                                           None, case["limit"], case["cap"], out, skip=state["skip"], layer=state["store"])
    if case["shared"]:
        return moe.moe_forward(state["store"], state["x"], state["ids"], state["w"], shared_expert=E)
    return exl3.apply_exl3_fused_moe(state["x"], state["ids"], state["w"], state["store"], None, None, case["limit"])


# ------------------------------------------------------------------------------------------------- what it takes

def work(case):
    H, I, k = SHAPES[case["shape"]]
    T = case["tokens"]
    if case["kind"] == "router":
        return {"bytes": T * H * 2 + E * H * 4 + T * E * 4 + T * k * 12, "flops": 2.0 * T * E * H}
    expert = 3 * H * I * 3 // 8 + (3 * H + 3 * I) * 2
    ids, _ = _routing(case, _gen(1, "cpu"), "cpu")
    counts = torch.bincount(ids.reshape(-1), minlength=E)
    if case["kind"] == "sorted":
        mean = float(counts[counts > case["cap"]].float().mean())
        routes, experts = mean * case["experts"], case["experts"]
    else:
        more = case["kind"] == "layers" or case["shared"]
        routes, experts = T * (k + 1 if more else k), int((counts > 0).sum()) + (1 if more else 0)
    x = T * H * torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    times = case.get("layers", 1)
    return {"bytes": times * (experts * expert + x + T * H * 4 + routes * 12), "flops": times * routes * 6.0 * H * I}


def tolerance(case):
    # router: fp32 sums of 4,096 or 5,120 products, and picks that may change places where two logits lie that close
    if case["kind"] == "router":
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
    # experts: fp16 activations at five points of each expert (transformed inputs, the three matrices' outputs before
    # and after their transforms, the activation), fp32 sums; weights rounded to fp16 or not: 5e-4 to 8e-4 off exact()
    return {"rel": 3e-3, "max": 4e-2}


# ------------------------------------------------------------------------------------------------- in 64 bits

_MUL1 = 0x83DCD12D
_KINV, _KBIAS = (float(np.array([b], np.uint16).view(np.float16)[0]) for b in (0x1EEE, 0xC931))


def _dense64(trellis, rounded):
    """fp64 [K, N] weights of a trellis [K/16, N/16, 48] int16: state i of a tile is the 16 bits ending at bit 3 i + 2 of
    its 768-bit stream (most significant bit first over 24 dwords), its weight KINV (1024 + byte sum of state x MUL1)
    + KBIAS, and it belongs to row 2 ((i >> 3) & 3) + (i & 1) + 8 ((i >> 1) & 1), column (i >> 5) + 8 ((i >> 2) & 1)."""
    kt, nt, _ = trellis.shape
    d = trellis.contiguous().view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    i = torch.arange(256, device=d.device)
    end = 3 * i + 2
    b = end >> 5
    s = (((d[..., (b + 23) % 24] << 32) | d[..., b]) >> (31 - (end & 31))) & 0xFFFF
    p = (s * _MUL1) & 0xFFFFFFFF
    s = (p & 255) + ((p >> 8) & 255) + ((p >> 16) & 255) + (p >> 24)
    w = _KINV * (1024 + s).double() + _KBIAS
    if rounded:
        w = w.half().double()
    at = torch.empty(256, dtype=torch.long, device=d.device)
    at[(2 * ((i >> 3) & 3) + (i & 1) + 8 * ((i >> 1) & 1)) * 16 + (i >> 5) + 8 * ((i >> 2) & 1)] = i
    return w[..., at].view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(kt * 16, nt * 16)


def _had64(x):
    """x [.., 128 m] times the orthonormal 128-point Hadamard matrix, block by block."""
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ (h / math.sqrt(128.0))).view(x.shape)


def _layer64(st, x, ids, w, limit, rounded, experts=None):
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in (torch.unique(ids).tolist() if experts is None else experts):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        if t.numel() == 0:
            continue
        xe = x[t]
        h = []
        for m in range(2):
            y = _had64(xe * st.w13_suh[e, m].double()) @ _dense64(st.w13_trellis[e, m], rounded)
            h.append(_had64(y) * st.w13_svh[e, m].double())
        a, u = h[0] * torch.sigmoid(h[0]), h[1]
        if limit > 0:
            a, u = a.clamp(max=limit), u.clamp(-limit, limit)
        y = _had64(a * u * st.w2_suh[e].double()) @ _dense64(st.w2_trellis[e], rounded)
        out.index_add_(0, t, _had64(y) * st.w2_svh[e].double() * w[t, j].double()[:, None])
    return out


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "router":
        logits = s["x"].double() @ s["gate"].double().t()
        v, ids = torch.topk(logits, SHAPES[case["shape"]][2], dim=1)
        return {"logits": logits, "ids": ids, "w": torch.softmax(v, 1)}
    rounded = bool(case.get("rounded", False))
    if case["kind"] == "layers":
        outs = []
        for st, x, ids, w in zip(s["stores"], s["x"], s["ids"], s["w"]):
            x = x.double()
            if case["rescale"]:
                x = x / x.square().mean(1, keepdim=True).sqrt()
            if case["dtype"] == "f32":
                x = x.bfloat16().double()                # an fp32 input is taken through bf16
            outs.append(_layer64(st, x, ids, w, case["limit"], rounded))
        return outs
    x, ids, w = s["x"].double(), s["ids"], s["w"]
    if case["kind"] == "sorted":
        experts = [e for e in s["batch"] if s["counts"][e] > case["cap"]]
        return _layer64(s["store"], x, ids, w.half(), case["limit"], rounded, experts)
    if case["shared"]:
        ids = torch.cat([ids, torch.full_like(ids[:, :1], E)], 1)
        w = torch.cat([w, torch.ones_like(w[:, :1])], 1)
    else:
        w = w.half()                                     # the plugin's routing weights are fp16
    return _layer64(s["store"], x, ids, w, case["limit"], rounded)
