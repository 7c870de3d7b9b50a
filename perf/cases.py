"""Performance cases of the full-attention path: what a program that drives it calls, step by step.

Every case is one call, or one layer's or one decode step's sequence of calls, through the package's public
functions. Five kinds:

  attention  the attention node of `layers` layers in one step, each over its own q4_0 K and V cache. form "mask"
             fills the step's F16 causal mask on the device and hands it to flash_attn_ext over the cache padded to
             256 rows (the engine's node); "causal" and "gate" are the mask-free entry point over the rows in use,
             without and with the fused output gate.
  layer      one full-attention layer as a step runs it: K and Q producers (RMSNorm, rotary, K quantized into the
             cache), V quantized on write, causal attention, gated W_o projection.
  append     KvCache.append of one step's K and V rows.
  out_proj   the gated W_o projection alone.

A step has `n` new tokens after `past` cached ones. The workspace and the outputs are kept by the caller, as a
serving loop keeps them.
"""
import math

import torch

import __graft_entry__ as graft

sqa = graft.load_package()

D = 256        # head dim of the attention kernels
N_EMBD = 2048  # width of the W_o output
N_ROT, SECTIONS, FREQ_BASE, EPS = 64, (11, 11, 10, 0), 1e7, 1e-6
MOST_PAIRS = 2048 * 132096 * 16  # (query row, key) pairs of the largest listed attention case


def listed():
    def attention(name, n, past, form, layers, H=16, Hkv=2):
        return {"name": name, "kind": "attention", "n": n, "past": past, "form": form, "layers": layers, "H": H, "Hkv": Hkv}

    return [
        # one decode step's node in a short conversation: launches and latency are everything
        attention("decode_4k_1layer", 1, 4095, "mask", 1),
        # a whole decode step's attention at a long context: ten layers' caches, 991 MB, more than any cache holds
        attention("decode_172k_10layers", 1, 172031, "mask", 10),
        # speculative verify of two positions at an ordinary context, all ten layers
        attention("verify2_32k_10layers", 2, 32766, "mask", 10),
        # the last, ragged chunk of a prompt or a short new message after a longer conversation
        attention("chunk37_after_20011_gate", 37, 20011, "gate", 1),
        # the first chunk of a prompt
        attention("chunk512_first", 512, 0, "mask", 1),
        # an ordinary chunk in the middle of a long prompt
        attention("chunk512_after_16384", 512, 16384, "mask", 1),
        # the largest ubatch at a long context, mask-free and gated
        attention("chunk2048_after_131072_gate", 2048, 131072, "gate", 1),
        # one layer of a decode step from the projections to the residual add
        {"name": "layer_decode_9001", "kind": "layer", "n": 1, "past": 9001, "H": 16, "Hkv": 2},
        # one layer of a ragged prompt chunk
        {"name": "layer_chunk300_after_3001", "kind": "layer", "n": 300, "past": 3001, "H": 16, "Hkv": 2},
        # the cache write of a prompt chunk whose norms and rotary stay in the caller's graph
        {"name": "append_512", "kind": "append", "n": 512, "past": 16384, "Hkv": 2},
        # W_o of a short message and of a prompt chunk
        {"name": "out_proj_23", "kind": "out_proj", "n": 23, "H": 16, "N": N_EMBD},
        {"name": "out_proj_512", "kind": "out_proj", "n": 512, "H": 16, "N": N_EMBD},
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))

    H, Hkv = rng.choice([(16, 2), (16, 2), (16, 2), (16, 4), (8, 2), (8, 1), (4, 4)])
    kind = rng.choice(["attention"] * 5 + ["layer", "append", "out_proj", "out_proj"])
    if kind == "append":
        return {"kind": kind, "n": log(1, 2048), "past": log(1, 131072) - 1, "Hkv": Hkv}
    if kind == "out_proj":
        return {"kind": kind, "n": log(1, 2048), "H": H, "N": rng.choice([1024, N_EMBD, N_EMBD, 4096, 16 * rng.randint(40, 320)])}
    n = rng.choice([1, 1, 2, rng.randint(3, 4)]) if rng.random() < 0.4 else log(5, 2048)
    past = log(64, 172032) if rng.random() < 0.85 else 0
    past = max(0, min(past, MOST_PAIRS // (n * H) - n))
    if kind == "layer":
        return {"kind": kind, "n": n, "past": min(past, 65536), "H": H, "Hkv": Hkv}
    return {"kind": kind, "n": n, "past": past, "form": rng.choice(["mask", "mask", "causal", "gate"]),
            "layers": rng.choice([1, 10]) if n <= 4 else 1, "H": H, "Hkv": Hkv}


# ------------------------------------------------------------------ inputs --

def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _q4_0(x):
    """Rows of q4_0 blocks of float32 rows: d = (value of largest magnitude) / -8 as fp16, codes
    min(15, int(x / d + 8.5)), 16 bytes with value j in the low nibble of byte j and j + 16 in its high one."""
    b = x.reshape(-1, 32)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    d = top / -8.0
    inv = torch.where(d != 0, torch.ones_like(d) / d, torch.zeros_like(d))
    y = b * inv
    y = y + 8.5
    c = y.to(torch.int32).clamp_(max=15).to(torch.uint8)
    out = torch.empty((b.shape[0], 18), dtype=torch.uint8, device=x.device)
    out[:, :2] = d.to(torch.float16).view(torch.uint8)
    out[:, 2:] = c[:, :16] | (c[:, 16:] << 4)
    return out.reshape(x.shape[0], -1)


def _cache(gen, rows, total, Hkv):
    """q4_0 cache of `total` rows, the first `rows` from N(0, 1), the others zero."""
    c = torch.zeros((total, Hkv * D // 32 * 18), dtype=torch.uint8, device="cuda")
    for r in range(0, rows, 32768):
        n = min(32768, rows - r)
        c[r:r + n] = _q4_0(_randn(gen, n, Hkv * D))
    return c.view(total, Hkv, D // 32 * 18)


def _q4_K(gen, N, K):
    """Q4_K weight rows: random codes and 6-bit scale and min pairs, fp16 d and dmin that centre the weights on 0."""
    w = torch.randint(0, 256, (N, K // 256, 144), generator=gen, device="cuda", dtype=torch.uint8)
    dm = torch.rand((N, K // 256, 2), generator=gen, device="cuda") * 4e-4 + 1e-4
    dm[:, :, 1] *= 7.5
    w[:, :, :4] = dm.to(torch.float16).view(torch.uint8).reshape(N, K // 256, 4)
    return w.reshape(N, -1)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _pad(n):
    return (n + 255) // 256 * 256


def _inputs(case, seed):
    g, kind, n = _gen(seed), case["kind"], case["n"]
    s = {"case": dict(case)}
    if kind == "out_proj":
        K = case["H"] * D
        return dict(s, w=_q4_K(g, case["N"], K), x=_randn(g, n, K), gate=_randn(g, n, K))
    past, Hkv = case["past"], case["Hkv"]
    if kind == "append":
        return dict(s, kc=_cache(g, past, _pad(past + n), Hkv), vc=_cache(g, past, _pad(past + n), Hkv),
                    k=_randn(g, n, Hkv * D), v=_randn(g, n, Hkv * D))
    H = case["H"]
    if kind == "layer":
        s.update(kc=_cache(g, past, _pad(past + n), Hkv), vc=_cache(g, past, _pad(past + n), Hkv),
                 k=_randn(g, n, Hkv, D), v=_randn(g, n, Hkv * D), q=_randn(g, n, H, D), gate=_randn(g, n, H * D),
                 kw=1 + 0.1 * _randn(g, D), qw=1 + 0.1 * _randn(g, D), w=_q4_K(g, N_EMBD, H * D))
        return s
    total = _pad(past + n) if case["form"] == "mask" else past + n
    s["kc"] = [_cache(g, past + n, total, Hkv) for _ in range(case["layers"])]
    s["vc"] = [_cache(g, past + n, total, Hkv) for _ in range(case["layers"])]
    s["q"] = [_randn(g, n, H, D) for _ in range(case["layers"])]
    if case["form"] == "gate":
        s["gate"] = [_randn(g, n, H, D) for _ in range(case["layers"])]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, n = case["kind"], case["n"]
    empty = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device="cuda")
    if kind == "out_proj":
        s.update(out=empty(n, case["N"]), ws=empty(max(1, sqa.out_proj_workspace_size(s["w"], s["x"])), dtype=torch.uint8))
    elif kind == "append":
        kv = sqa.KvCache(1, D, case["Hkv"], case["past"] + n)
        kv.k[0].copy_(s.pop("kc"))
        kv.v[0].copy_(s.pop("vc"))
        kv.begin_step(case["past"])
        s.update(kv=kv, idx=torch.arange(case["past"], case["past"] + n, device="cuda", dtype=torch.int64))
    elif kind == "layer":
        H, past = case["H"], case["past"]
        s["idx"] = torch.arange(past, past + n, device="cuda", dtype=torch.int64)
        s["pos"] = torch.arange(past, past + n, device="cuda", dtype=torch.int32).repeat(4)
        s["rope"] = sqa.rope_params(N_ROT, SECTIONS, FREQ_BASE)
        s.update(q_rot=empty(n, H, D), attn=empty(n, H, D), out=empty(n, N_EMBD))
        need = max(sqa.flash_attn_workspace_size(s["q_rot"], s["kc"], past + n),
                   sqa.out_proj_workspace_size(s["w"], s["attn"].view(n, H * D)))
        s["ws"] = empty(need, dtype=torch.uint8)
    else:
        s["out"] = [torch.empty_like(q) for q in s["q"]]
        n_kv = s["kc"][0].shape[0]
        s["ws"] = empty(sqa.flash_attn_workspace_size(s["q"][0], s["kc"][0], n_kv), dtype=torch.uint8)
        if case["form"] == "mask":
            s["mask"] = empty(n, n_kv, dtype=torch.float16)
    return s


def run(s):
    case = s["case"]
    kind, n = case["kind"], case["n"]
    if kind == "out_proj":
        return sqa.out_proj(s["w"], s["x"], gate=s["gate"], out=s["out"], workspace=s["ws"])
    past = case["past"]
    if kind == "append":
        kv = s["kv"]
        kv.rewind_to(past)
        kv.begin_step(n)
        kv.append(0, s["k"], s["v"], s["idx"])
        return kv.k[0], kv.v[0]
    if kind == "layer":
        kc, vc, flat = s["kc"], s["vc"], (n, case["H"] * D)
        sqa.rope_norm_set_rows_q4_0(kc, s["k"], s["kw"], EPS, s["pos"], s["rope"], s["idx"])
        sqa.set_rows_q4_0(vc, s["v"], s["idx"])
        sqa.rope_norm_f32(s["q_rot"], s["q"], s["qw"], EPS, s["pos"], s["rope"])
        sqa.flash_attn_ext_causal(s["q_rot"], kc, vc, past + n, past, out=s["attn"], workspace=s["ws"])
        sqa.out_proj(s["w"], s["attn"].view(flat), gate=s["gate"], out=s["out"], workspace=s["ws"])
        return {"out": s["out"], "attn": s["attn"], "q": s["q_rot"], "k": kc, "v": vc}
    n_kv = s["kc"][0].shape[0]
    if case["form"] == "mask":
        sqa.fill_causal_mask(s["mask"], past)
    for i in range(case["layers"]):
        a = (s["q"][i], s["kc"][i], s["vc"][i], n_kv)
        if case["form"] == "mask":
            sqa.flash_attn_ext(*a, mask=s["mask"], out=s["out"][i], workspace=s["ws"])
        else:
            sqa.flash_attn_ext_causal(*a, past, gate=s["gate"][i] if "gate" in s else None, out=s["out"][i],
                                      workspace=s["ws"])
    return s["out"]


def work(case):
    n, kind = case["n"], case["kind"]
    if kind == "out_proj":
        K, N = case["H"] * D, case["N"]
        return {"bytes": N * K // 256 * 144 + n * (2 * K + N) * 4, "flops": 2 * n * N * K}
    row = case["Hkv"] * D // 32 * 18  # bytes of one cache row
    write = n * 2 * (case["Hkv"] * D * 4 + row)
    if kind == "append":
        return {"bytes": write, "flops": 0}
    past, H = case["past"], case["H"]
    pairs = n * past + n * (n + 1) // 2
    read, qo, attn = (past + n) * 2 * row, n * H * D * 4, 4 * D * H * pairs
    if kind == "layer":
        proj = work({"kind": "out_proj", "n": n, "H": H, "N": N_EMBD})
        return {"bytes": write + read + 4 * qo + proj["bytes"], "flops": attn + proj["flops"]}
    # the mask is read where it is the entry point's input: once, the same for every layer
    mask = 2 * n * (past + n) if case["form"] == "mask" else 0
    return {"bytes": case["layers"] * (read + (3 if case["form"] == "gate" else 2) * qo) + mask,
            "flops": case["layers"] * attn}


def tolerance(case):
    # about four times the largest distance to the 64-bit results seen over listed and drawn cases of each kind:
    # attention 3.9e-6, W_o 2.5e-6, layer 1.8e-5 (a value an ulp off may round to the neighbouring q8_0 or q4_0 code)
    if case["kind"] == "append":
        return "exact"
    if case["kind"] == "out_proj":
        return {"rel": 1e-5}
    if case["kind"] == "layer":
        return {"rel": 7e-5, "max": 1e-2, "differ": 1e-5}
    return {"rel": 1.6e-5}


# --------------------------------------------------- the same in 64 bits --

def _from_q4_0(cache):
    """float64 (rows, Hkv, D) of a q4_0 cache."""
    rows, Hkv, _ = cache.shape
    b = cache.reshape(-1, 18)
    d = b[:, :2].contiguous().view(torch.float16).to(torch.float64)
    c = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(torch.float64)
    return ((c - 8) * d).view(rows, Hkv, D)


def _q8_0(q):
    """The values of float32 rows rounded to q8_0 (d = amax / 127 as fp16, codes rint(x * 127 / amax)), as float64."""
    b = q.reshape(-1, 32)
    amax = b.abs().amax(1, keepdim=True)
    top = torch.full_like(amax, 127.0)  # a tensor: torch divides by a plain number through its reciprocal
    d = (amax / top).to(torch.float16).to(torch.float64)
    inv = torch.where(amax != 0, top / amax, torch.zeros_like(amax))
    return (torch.round(b * inv).to(torch.float64) * d).view(q.shape)


def _attention(q, kc, vc, past, gate=None):
    n, H, _ = q.shape
    n_kv, G = past + n, H // kc.shape[1]
    k, v, qd = _from_q4_0(kc[:n_kv]), _from_q4_0(vc[:n_kv]), _q8_0(q)
    out = torch.empty((n, H, D), dtype=torch.float64, device=q.device)
    last = past + torch.arange(n, device=q.device)
    for h in range(H):
        for r in range(0, n, 512):
            s = qd[r:r + 512, h] @ k[:, h // G].t() * D ** -0.5
            s.masked_fill_(torch.arange(n_kv, device=q.device) > last[r:r + 512, None], -math.inf)
            out[r:r + 512, h] = torch.softmax(s, 1) @ v[:, h // G]
    return out if gate is None else out * torch.sigmoid(gate.double())


def _project(w, x, gate):
    N = w.shape[0]
    b = w.view(N, -1, 144)
    dm = b[:, :, :4].contiguous().view(torch.float16).to(torch.float64)
    q = b[:, :, 4:16].to(torch.int32)
    sc = torch.cat([q[..., :4] & 63, (q[..., 8:] & 15) | (q[..., :4] >> 6 << 4)], -1)
    mn = torch.cat([q[..., 4:8] & 63, (q[..., 8:] >> 4) | (q[..., 4:8] >> 6 << 4)], -1)
    qs = b[:, :, 16:].reshape(N, -1, 4, 1, 32)
    codes = torch.cat([qs & 15, qs >> 4], 3).reshape(N, -1, 8, 32).to(torch.float64)
    wd = codes * (dm[..., :1] * sc)[..., None] - (dm[..., 1:] * mn)[..., None]
    return (x.double() * torch.sigmoid(gate.double())) @ wd.reshape(N, -1).t()


def _producer(x, w, pos):
    """RMSNorm times w, then the rotation of the first N_ROT dims; the four position components are equal, so every
    sector of the rotary sections turns by the same position."""
    x = x.double()
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    half = N_ROT // 2
    step = float(torch.tensor(FREQ_BASE, dtype=torch.float32) ** (-2.0 / N_ROT))
    angle = torch.empty((pos.shape[0], half), dtype=torch.float32, device=x.device)
    angle[:, 0] = pos.float()
    for i in range(1, half):  # the op defines the angle by float32 steps
        angle[:, i] = angle[:, i - 1] * step
    c, s = torch.cos(angle.double())[:, None], torch.sin(angle.double())[:, None]
    out = y.clone()
    out[..., :half] = y[..., :half] * c - y[..., half:N_ROT] * s
    out[..., half:N_ROT] = y[..., :half] * s + y[..., half:N_ROT] * c
    return out


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    s = _inputs(case, seed)
    if kind == "append":
        for c, x in ((s["kc"], s["k"]), (s["vc"], s["v"])):
            c[case["past"]:case["past"] + n] = _q4_0(x).view(n, *c.shape[1:])
        return s["kc"], s["vc"]
    if kind == "out_proj":
        return _project(s["w"], s["x"], s["gate"])
    past = case["past"]
    if kind == "layer":
        pos = torch.arange(past, past + n, device="cuda")
        q = _producer(s["q"], s["qw"], pos)
        s["kc"][past:past + n] = _q4_0(_producer(s["k"], s["kw"], pos).float().reshape(n, -1)).view(n, *s["kc"].shape[1:])
        s["vc"][past:past + n] = _q4_0(s["v"]).view(n, *s["vc"].shape[1:])
        attn = _attention(q.float(), s["kc"], s["vc"], past)
        return {"out": _project(s["w"], attn.reshape(n, -1), s["gate"]), "attn": attn, "q": q, "k": s["kc"], "v": s["vc"]}
    return [_attention(s["q"][i], s["kc"][i], s["vc"][i], past, s["gate"][i] if "gate" in s else None)
            for i in range(case["layers"])]
