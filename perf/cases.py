"""The work that programs give this package, as timed cases: the projections, the attention and the whole steps of a
batch-1 int4 decoder (hidden 2048, 16 query / 4 KV heads of 128, MLP 11008, 16385 audio logits, 2048 cache slots).

listed() and draw() give cases as dicts of plain values, prepare() a case's inputs, weights and plans on the GPU, run()
one pass through the package's entry points, work() what a pass cannot do without, tolerance() how far another correct
implementation may be off, exact() the same outputs in 64 bits from plain torch.

A case with "layers" > 1 is a chain over that many weight sets, as a decoder walks its layers; it is captured once in
a hipGraph and a pass is one replay, as the engines run it. The others call the entry point eagerly.
"""
import math
import sys
from pathlib import Path

import torch

PKG = Path(__file__).resolve().parents[1] / "rumik-fast_amd"
for _p in (PKG / "kernels", PKG / "engine"):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

import cuda_gemv  # noqa: E402
import decode  # noqa: E402
import fused  # noqa: E402
import mm_int4  # noqa: E402
import prefill  # noqa: E402

DEV = "cuda"
G = 128
H, NH, HD, INTER, SLOTS, AUDIO, VOCAB = 2048, 16, 128, 11008, 2048, 16385, 4096
NKV = 4
N_PLAIN = (NH + 2 * NKV) * HD          # q | k | v rows of the input projection
N_IN = N_PLAIN + 2 * INTER             # with the gate and up rows: 25088
EPS, THETA = 1e-5, 10000.0
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # the smallest call: one output projection of a decode step, called by itself (the drop-in GEMV)
        {"name": "gemv_o", "kind": "gemv", "N": 2048, "K": 2048, "dtype": "fp16", "layers": 1},
        # the projections of a decode step as a launch-per-kernel engine runs them over its layers: the fused input
        # projection with SiLU(gate) * up, then the output and down projections together
        {"name": "gemv_layers", "kind": "gemv_layers", "inter": 11008, "dtype": "bf16", "layers": 12},
        # the audio head of one token: int8 rows, fp32 logits
        {"name": "head", "kind": "head", "N": 16385, "K": 2048, "dtype": "fp16"},
        # decode attention halfway through the cache, over the layers of the launch-per-kernel engine
        {"name": "attn_1000", "kind": "attn", "ctx": 1000, "nkv": 4, "dtype": "bf16", "layers": 12},
        # the input projection of a short prompt (34 tokens: the usual sentence)
        {"name": "mm_in_34", "kind": "mm", "T": 34, "N": 25088, "K": 2048, "dtype": "bf16", "layers": 6},
        # the output projection of a 69-token prompt: few columns, ragged rows
        {"name": "mm_o_69", "kind": "mm", "T": 69, "N": 2048, "K": 2048, "dtype": "fp16", "layers": 12},
        # the down projection of a 200-token prompt: long rows, few columns
        {"name": "mm_down_200", "kind": "mm", "T": 200, "N": 2048, "K": 11008, "dtype": "bf16", "layers": 6},
        # the input projection of a long prompt (512 tokens), called by itself
        {"name": "mm_in_512", "kind": "mm", "T": 512, "N": 25088, "K": 2048, "dtype": "fp16", "layers": 1},
        # causal attention of a 512-token prompt over the layers
        {"name": "prefill_attn_512", "kind": "prefill_attn", "T": 512, "p0": 0, "nkv": 4, "layers": 6},
        # two decoder layers of the longest prompts (voice prompt and text): projections, attention and row kernels
        # with everything between them, launched eagerly as Prefill does by default
        {"name": "layers_1024", "kind": "prefill", "T": 1024, "L": 2, "graphs": False},
        # the whole prefill of a 69-token prompt through all 36 layers, replayed as a server does
        {"name": "prefill_69", "kind": "prefill", "T": 69, "L": 36, "graphs": True},
        # one token of the 36-layer model at position 300 with the sampling tail in the step
        {"name": "decode_300", "kind": "decode", "pos": 300, "L": 36},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv_layers", "head", "attn", "mm", "mm", "mm", "prefill_attn", "prefill", "decode"])
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "gemv":
        K = 128 * rng.randint(4, 86)
        N = min(_log(rng, 512, 25088), 25088 * 2048 // K)
        return {"kind": kind, "N": N, "K": K, "dtype": dtype, "layers": rng.choice([1, 8])}
    if kind == "gemv_layers":
        return {"kind": kind, "inter": 128 * rng.randint(16, 96), "dtype": dtype, "layers": rng.randint(6, 12)}
    if kind == "head":
        return {"kind": kind, "N": _log(rng, 1000, 16385), "K": 2048, "dtype": dtype}
    if kind == "attn":
        return {"kind": kind, "ctx": _log(rng, 1, 2047), "nkv": rng.choice([4, 8]), "dtype": dtype, "layers": 12}
    if kind == "mm":
        T = _log(rng, 8, 512)
        if rng.random() < 0.6:
            N, K = rng.choice([(25088, 2048), (22016, 2048), (3072, 2048), (2048, 2048), (2048, 11008)])
        else:
            K = 128 * rng.randint(4, 86)
            N = min(_log(rng, 512, 25088), 25088 * 2048 // K)
        return {"kind": kind, "T": T, "N": N, "K": K, "dtype": dtype, "layers": rng.choice([1, 4])}
    if kind == "prefill_attn":
        T = _log(rng, 8, 1024)
        return {"kind": kind, "T": T, "p0": rng.choice([0, 0, rng.randint(1, 512)]), "nkv": rng.choice([4, 8]),
                "layers": 4}
    if kind == "prefill":
        return {"kind": kind, "T": _log(rng, 8, 1024), "L": rng.randint(1, 2), "graphs": rng.choice([True, False])}
    return {"kind": kind, "pos": _log(rng, 1, 2040), "L": rng.choice([2, 4, 8])}


# ---------------------------------------------------------------------------------------------- inputs from a seed
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _int4(g, n, k):
    """codes uniform in 0..15, scale ~ U[1e-3, 2e-2], min = (-7.5 + N(0, 1)) * scale per 128 columns"""
    q = torch.randint(0, 256, (n, k // 2), generator=g, device=DEV, dtype=torch.uint8)
    s = (torch.rand(n, k // G, generator=g, device=DEV) * 1.9e-2 + 1e-3).half()
    m = ((torch.randn(n, k // G, generator=g, device=DEV) - 7.5) * s.float()).half()
    return q, s, m


def _int8(g, n, k):
    q = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    return q, (torch.rand(n, generator=g, device=DEV) * 9e-3 + 1e-3).half()


def _normal(g, *shape, dtype=torch.float16):
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _ln(g):
    return (torch.rand(H, generator=g, device=DEV) + 0.5).half()


def _model(g, L):
    w = {"w_in": [], "w_o": [], "w_down": [], "ln": []}
    for _ in range(L):
        w["w_in"].append(_int4(g, N_IN, H))
        w["w_o"].append(_int4(g, H, H))
        w["w_down"].append(_int4(g, H, INTER))
        w["ln"].append(_ln(g))
    w["norm"], w["emb"], w["head"] = _ln(g), _int8(g, VOCAB, H), _int8(g, AUDIO, H)
    return w


def _stop(g):
    """the stop predictor's state dict (LayerNorm, 512 x 2048 GELU layer, one output)"""
    return {"0.weight": torch.ones(H, device=DEV), "0.bias": torch.zeros(H, device=DEV),
            "1.weight": _normal(g, 512, H, dtype=torch.float32).mul(H ** -0.5).bfloat16(),
            "1.bias": torch.zeros(512, device=DEV),
            "3.weight": _normal(g, 1, 512, dtype=torch.float32).mul(512 ** -0.5).bfloat16(),
            "3.bias": torch.full((1,), -4.0, device=DEV)}


def _inputs(c, seed):
    """Everything a case reads, from the seed alone (prepare() and exact() both start here)."""
    g = _gen(seed)
    kind, d = c["kind"], {}
    dt = DT[c.get("dtype", "fp16")]
    if kind in ("gemv", "mm"):
        d["w"] = [_int4(g, c["N"], c["K"]) for _ in range(c["layers"])]
        d["x"] = _normal(g, *((c["T"],) if kind == "mm" else ()), c["K"], dtype=dt)
    elif kind == "gemv_layers":
        n = c["inter"]
        d["w"] = [(_int4(g, N_PLAIN + 2 * n, H), _int4(g, H, H), _int4(g, H, n)) for _ in range(c["layers"])]
        d["x"], d["o"] = _normal(g, H, dtype=dt), _normal(g, H, dtype=dt)
    elif kind == "head":
        d["w"], d["x"] = _int8(g, c["N"], c["K"]), _normal(g, c["K"], dtype=dt)
    elif kind == "attn":
        d["q"] = _normal(g, c["layers"], NH * HD, dtype=dt)
        d["k"], d["v"] = (_normal(g, c["layers"], c["nkv"], SLOTS, HD, dtype=dt) for _ in range(2))
    elif kind == "prefill_attn":
        d["q"] = _normal(g, c["layers"], c["T"], NH * HD)
        d["k"], d["v"] = (_normal(g, c["layers"], c["nkv"], SLOTS, HD) for _ in range(2))
    elif kind == "prefill":
        d["w"] = _model(g, c["L"])
        d["ids"] = torch.randint(0, VOCAB, (c["T"],), generator=g, device=DEV).tolist()
    else:
        d["w"], d["stop"] = _model(g, c["L"]), _stop(g)
        d["tok"] = int(torch.randint(0, VOCAB, (1,), generator=g, device=DEV))
        d["k"], d["v"] = (_normal(g, c["L"], NKV, c["pos"], HD) for _ in range(2))
    return d


# ---------------------------------------------------------------------------------------------- a pass
def _config(L):
    return decode.Config(L=L, H=H, NH=NH, NKV=NKV, HD=HD, inter=INTER, S=SLOTS, n_audio=AUDIO, vocab=VOCAB, eps=EPS,
                         rope_theta=THETA)


def _captured(fn):
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    dt = DT[c.get("dtype", "fp16")]
    new = lambda *s, dtype=dt: torch.empty(*s, device=DEV, dtype=dtype)  # noqa: E731
    st = {"d": d, "kind": kind}
    if kind in ("gemv", "mm"):
        f = cuda_gemv.gemv_int4_cuda if kind == "gemv" else mm_int4.mm_int4
        rows = (c["T"],) if kind == "mm" else ()
        outs = [new(*rows, c["N"]) for _ in d["w"]]
        calls = [lambda w=w, y=y: f(d["x"], *w, out=y) for w, y in zip(d["w"], outs)]
    elif kind == "gemv_layers":
        n = c["inter"]
        outs = [{"y": new(N_PLAIN), "act": new(n), "o": new(H), "down": new(H)} for _ in d["w"]]

        def layer(w, y):
            cuda_gemv.gemv_int4_silu_cuda(d["x"], *w[0], N_PLAIN, out=y["y"], act=y["act"])
            cuda_gemv.gemv_int4_pair_cuda(d["o"], w[1], y["act"], w[2], out1=y["o"], out2=y["down"])

        calls = [lambda w=w, y=y: layer(w, y) for w, y in zip(d["w"], outs)]
    elif kind == "head":
        outs = new(c["N"], dtype=torch.float32)
        calls = [lambda: cuda_gemv.gemv_int8_cuda(d["x"], *d["w"], out=outs)]
    elif kind == "attn":
        nkv, ns = c["nkv"], 64
        outs = new(c["layers"], NH * HD)
        po = new(NH, ns, HD, dtype=torch.float32)
        pm, pl = new(NH, ns, dtype=torch.float32), new(NH, ns, dtype=torch.float32)
        pos = torch.full((1,), c["ctx"], device=DEV, dtype=torch.int64)  # slots 0 .. ctx

        def layer(i):
            fused.attn_split[(nkv, ns)](d["q"][i], d["k"][i], d["v"][i], pos, po, pm, pl, SLOTS, HD ** -0.5,
                                        REP=NH // nkv, HD=HD, NSPLIT=ns)
            fused.attn_combine[(NH,)](po, pm, pl, pos, outs[i], HD=HD, NSPLIT=ns)

        calls = [lambda i=i: layer(i) for i in range(c["layers"])]
    elif kind == "prefill_attn":
        outs = new(c["layers"], c["T"], NH * HD)
        calls = [lambda i=i: prefill.prefill_attn(d["q"][i], d["k"][i], d["v"][i], outs[i], c["T"], c["p0"], NH,
                                                  c["nkv"], HD, SLOTS, HD ** -0.5) for i in range(c["layers"])]
    elif kind == "prefill":
        cfg = _config(c["L"])
        kc, vc = (torch.zeros(c["L"], NKV, SLOTS, HD, device=DEV, dtype=torch.float16) for _ in range(2))
        cos, sin = decode.rope_tables(SLOTS, HD, THETA, torch.float16, DEV)
        st["pf"] = prefill.Prefill(cfg, d["w"], kc, vc, cos, sin, max_T=1024, graphs=c["graphs"])
        st["hn"] = new(H)
        st["pf"].run(d["ids"])  # the first prompt of a length bucket captures its graph: once, when a server starts
        return st
    else:
        eng = decode.RoleDecode(_config(c["L"]), d["w"], device=torch.device(DEV, torch.cuda.current_device()))
        eng.kc[:, :, :c["pos"]] = d.pop("k")
        eng.vc[:, :, :c["pos"]] = d.pop("v")
        ids = torch.arange(AUDIO, device=DEV) % (VOCAB - 1)
        ids[-1] = VOCAB - 1  # </audio>, on exactly one row
        eng.attach_sampler(d["stop"], ids, VOCAB - 1, max_new=64)
        eng.set_state(d["tok"], c["pos"])
        eng.capture()
        st.update(eng=eng, pos=c["pos"])
        return st
    st["outs"] = outs
    if len(calls) == 1:
        st["call"] = calls[0]
    else:
        def chain():
            for f in calls:
                f()

        st["graph"] = _captured(chain)
        st["held"] = calls  # the graph holds addresses only: everything the calls use lives as long as the state
        st["call"] = st["graph"].replay
    return st


def run(st):
    kind = st["kind"]
    if kind == "prefill":
        st["pf"].run(st["d"]["ids"], hn=st["hn"])
        T = len(st["d"]["ids"])
        return {"hn": st["hn"], "k": st["pf"].kc[:, :, :T], "v": st["pf"].vc[:, :, :T]}
    if kind == "decode":
        # one replay from this position, as the teacher-forced prompt loop runs it: the token sampled from these
        # logits is random by design and is not an output here
        e, pos = st["eng"], st["pos"]
        e.set_state(st["d"]["tok"], pos)
        e.step_i.zero_()
        e.replay()
        return {"logits": e.logits, "hn": e.hn, "k": e.kc[:, :, pos], "v": e.vc[:, :, pos], "stop": e.sampler.z1}
    st["call"]()
    return st["outs"]


# ---------------------------------------------------------------------------------------------- what a pass needs
def _i4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // G)


def _layer_bytes():
    return _i4_bytes(N_IN, H) + _i4_bytes(H, H) + _i4_bytes(H, INTER)


def work(case):
    c = case
    kind, n = c["kind"], c.get("layers", 1)
    if kind in ("gemv", "mm"):
        T = c.get("T", 1)
        return {"bytes": n * (_i4_bytes(c["N"], c["K"]) + 2 * T * c["N"]) + 2 * T * c["K"],
                "flops": 2 * n * T * c["N"] * c["K"]}
    if kind == "gemv_layers":
        i = c["inter"]
        sizes = ((N_PLAIN + 2 * i, H), (H, H), (H, i))
        return {"bytes": n * (sum(_i4_bytes(*s) for s in sizes) + 2 * (N_PLAIN + i + 2 * H)) + 4 * H,
                "flops": 2 * n * sum(a * b for a, b in sizes)}
    if kind == "head":
        return {"bytes": c["N"] * c["K"] + 2 * c["N"] + 2 * c["K"] + 4 * c["N"], "flops": 2 * c["N"] * c["K"]}
    if kind == "attn":
        return {"bytes": n * (4 * c["nkv"] * (c["ctx"] + 1) * HD + 4 * NH * HD), "flops": 4 * n * NH * (c["ctx"] + 1) * HD}
    if kind == "prefill_attn":
        T, p0 = c["T"], c["p0"]
        return {"bytes": n * (4 * T * NH * HD + 4 * c["nkv"] * (p0 + T) * HD),
                "flops": 4 * n * NH * HD * (T * p0 + T * (T + 1) // 2)}
    if kind == "prefill":
        T, L = c["T"], c["L"]
        mm = 2 * T * (N_IN * H + H * H + H * INTER)
        return {"bytes": L * (_layer_bytes() + 4 * NKV * T * HD + 2 * H) + T * (H + 10) + 4 * H,
                "flops": L * (mm + 2 * NH * HD * T * (T + 1))}
    L, pos = c["L"], c["pos"]
    return {"bytes": L * (_layer_bytes() + 4 * NKV * (pos + 1) * HD + 2 * H) + AUDIO * (H + 6) + 512 * H * 2 + 6 * H,
            "flops": 2 * L * (N_IN * H + H * H + H * INTER) + 4 * L * NH * (pos + 1) * HD + 2 * AUDIO * H + 1024 * H}


def tolerance(case):
    # Against 64 bits, measured: one 16-bit rounding of an fp32 sum is 2.1e-4 (fp16) or 1.7e-3 (bf16); down over the
    # rounded activation 3.6e-3 in bf16; the prefill attention, with fp16 weights of V, 2.4e-4; the head's fp32
    # logits 7.6e-8; whole steps 1.1e-3 after 2 layers, 2e-3 after 4, 6.4e-3 after 36. Four times each (the logits
    # more: another order of 2048 additions).
    c = case
    kind = c["kind"]
    if kind == "head":
        return {"rel": 1e-6, "max": 4e-5}
    if kind in ("prefill", "decode"):
        rel = 5e-3 * max(1.0, c["L"] / 2) ** 0.57
        return {"rel": rel, "max": 20 * rel}
    if kind == "prefill_attn":
        return {"rel": 1e-3, "max": 0.03}
    fp16 = c["dtype"] == "fp16"
    if kind == "gemv_layers":
        return {"rel": 1.8e-3 if fp16 else 1.4e-2, "max": 0.04 if fp16 else 0.3}
    return {"rel": 8e-4 if fp16 else 7e-3, "max": 0.03 if fp16 else 0.25}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _deq(w):
    q, s, m = w
    codes = torch.stack((q & 15, q >> 4), dim=-1).reshape(q.shape[0], -1, G).double()
    return (codes * s.double().unsqueeze(-1) + m.double().unsqueeze(-1)).reshape(q.shape[0], -1)


def _layernorm(x, w):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, p0):
    """x [T, heads, HD] at positions p0 .. p0 + T - 1, interleaved pairs, the engine's fp16 tables"""
    inv = 1.0 / (THETA ** (torch.arange(0, HD, 2, dtype=torch.float32) / HD))
    a = torch.outer(torch.arange(SLOTS, dtype=torch.float32), inv)[p0:p0 + x.shape[0]]
    cos, sin = a.cos().half().to(DEV).double()[:, None], a.sin().half().to(DEV).double()[:, None]
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * cos - o * sin, o * cos + e * sin), dim=-1).flatten(-2)


def _attend(q, k, v, p0):
    """q [T, NH, HD] at positions p0 .., k / v [nkv, >= p0 + T, HD] -> [T, NH * HD], causal"""
    T, n, rep = q.shape[0], p0 + q.shape[0], NH // k.shape[0]
    mask = torch.arange(n, device=DEV)[None] > (p0 + torch.arange(T, device=DEV))[:, None]
    out = torch.empty(T, NH, HD, device=DEV, dtype=torch.float64)
    for h in range(NH):
        s = (q[:, h].contiguous() @ k[h // rep, :n].double().t().contiguous()) * HD ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[h // rep, :n].double()
    return out.reshape(T, NH * HD)


def _mlp_act(y):
    gate, up = y[..., N_PLAIN:].chunk(2, -1)
    return gate / (1 + torch.exp(-gate)) * up


def _layers(w, ids, p0, past=None):
    """The decoder over tokens at positions p0 ..: (final LayerNorm [T, H], k, v [L, NKV, T, HD])"""
    L, T = len(w["w_in"]), len(ids)
    ids = torch.tensor(ids, device=DEV)
    x = w["emb"][0][ids].double() * w["emb"][1][ids].double()[:, None]
    ks, vs = [], []
    for i in range(L):
        h = _layernorm(x, w["ln"][i])
        y = h @ _deq(w["w_in"][i]).t()
        q, k, v = (t.reshape(T, -1, HD) for t in y[:, :N_PLAIN].split([NH * HD, NKV * HD, NKV * HD], -1))
        if i % 4 != 3:  # three of every four layers rotate
            q, k = _rope(q, p0), _rope(k, p0)
        k, v = k.transpose(0, 1), v.transpose(0, 1)
        ks.append(k)
        vs.append(v)
        if past is not None:
            k, v = torch.cat((past[0][i].double(), k), 1), torch.cat((past[1][i].double(), v), 1)
        x = x + _attend(q, k, v, p0) @ _deq(w["w_o"][i]).t() + _mlp_act(y) @ _deq(w["w_down"][i]).t()
    return _layernorm(x, w["norm"]), torch.stack(ks), torch.stack(vs)


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    if kind in ("gemv", "mm"):
        return [d["x"].double() @ _deq(w).t() for w in d["w"]]
    if kind == "gemv_layers":
        outs = []
        for w_in, w_o, w_down in d["w"]:
            y = d["x"].double() @ _deq(w_in).t()
            act = _mlp_act(y)
            outs.append({"y": y[:N_PLAIN], "act": act, "o": d["o"].double() @ _deq(w_o).t(),
                         "down": act @ _deq(w_down).t()})
        return outs
    if kind == "head":
        return (d["w"][0].double() @ d["x"].double()) * d["w"][1].double()
    if kind in ("attn", "prefill_attn"):
        T, p0 = c.get("T", 1), c.get("p0", c.get("ctx"))
        o = [_attend(d["q"][i].double().reshape(T, NH, HD), d["k"][i], d["v"][i], p0) for i in range(c["layers"])]
        return torch.stack(o).reshape(c["layers"], -1) if kind == "attn" else torch.stack(o)
    if kind == "prefill":
        h, k, v = _layers(d["w"], d["ids"], 0)
        return {"hn": h[-1], "k": k, "v": v}
    h, k, v = _layers(d["w"], [d["tok"]], c["pos"], (d["k"], d["v"]))
    h, s = h[0], d["stop"]
    n = h - h.mean()
    n = n / torch.sqrt((n * n).mean() + 1e-5) * s["0.weight"].double() + s["0.bias"].double()
    z = s["1.weight"].double() @ n + s["1.bias"].double()
    return {"logits": (d["w"]["head"][0].double() @ h) * d["w"]["head"][1].double(), "hn": h, "k": k[:, :, 0],
            "v": v[:, :, 0], "stop": 0.5 * z * (1 + torch.erf(z / math.sqrt(2)))}
