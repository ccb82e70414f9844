"""The calls that an engine on top of this library spends its time in, at the
sizes of the 8B configuration (hidden 4096, MLP 12800, 32 query and 8 KV heads
of 128, vocabulary 100352), over the ranges an engine meets: one token to a
chunk of 8192 tokens, contexts up to 65536 positions, every KV pool format,
FP8 and bf16 activations.

Each case is a dict; `listed` gives the standing ones, `draw` another one of
the same ranges. `prepare` makes what an engine holds before the call (inputs,
weights, pool, plan), `run` makes one pass through the entry points, `work` says
what a pass cannot do without, `exact` evaluates the same inputs in 64 bits and
`tolerance` says how far two correct implementations may be apart.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

H, INTER, HQ, HK, D, VOCAB = 4096, 12800, 32, 8, 128, 100352
NQ, NK = HQ * D, HK * D
MAX_POS = 65536
EPS = 1e-5
RESID, EMB_MULT, ATTN_SCALE, THETA = 0.22, 12.0, 1.0 / 128, 1e7
W_STD = 80.0  # std of the e4m3 weight codes: normal weights under amax / 448

_L = None


def _layerops():
    global _L
    if _L is None:
        path = os.path.join(os.getcwd(), "granite-4-rtx-4070-ti-super_amd", "layerops.py")
        spec = importlib.util.spec_from_file_location("g4_layerops", path)
        _L = importlib.util.module_from_spec(spec)
        sys.modules["g4_layerops"] = _L
        spec.loader.exec_module(_L)
    return _L


# --------------------------------------------------------------------- cases
def listed():
    return [
        # one user's chat: the token loop's step at a few thousand tokens of
        # context (8 of the 40 layers and the LM head), replayed as one graph
        {"name": "token-step", "kind": "token", "layers": 8, "context": 4321, "bits": 16,
         "group": 128},
        # a server's batched step: 8 sessions anywhere in [0, 65536), int8 pool
        {"name": "session-step", "kind": "sessions", "layers": 2, "sessions": 8, "bits": 8,
         "fp8": True},
        # the non-GEMM ops of a layer: a batch of decode rows, a prompt, a long
        # chunk at the end of a long context
        {"name": "ops-8", "kind": "ops", "tokens": 8, "start": 1000, "bits": 8, "group": 128},
        {"name": "ops-512", "kind": "ops", "tokens": 512, "start": 0, "bits": 8, "group": 128},
        {"name": "ops-8192", "kind": "ops", "tokens": 8192, "start": 57344, "bits": 5,
         "group": 32},
        # decode attention of one session far into a document
        {"name": "attn-decode", "kind": "attn_decode", "rows": 1, "context": 30011, "bits": 8,
         "group": 128},
        # a short prompt's attention, and the last chunk of a 65536-token document's
        {"name": "attn-prompt", "kind": "attn_prefill", "tokens": 500, "start": 0, "bits": 8,
         "group": 128},
        {"name": "attn-document", "kind": "attn_prefill", "tokens": 8192, "start": 57344,
         "bits": 5, "group": 32},
        # the projections of a chunk with FP8 activations
        {"name": "gate-up-8192", "kind": "gemm", "proj": "gate_up", "tokens": 8192, "fp8": True},
        {"name": "down-512", "kind": "gemm", "proj": "down", "tokens": 512, "fp8": True},
        # and with the engine's bf16 activations: a prompt of ordinary, ragged
        # length, and the O projection of a full chunk
        {"name": "qkv-1000", "kind": "gemm", "proj": "qkv", "tokens": 1000, "fp8": False},
        {"name": "o-8192", "kind": "gemm", "proj": "o", "tokens": 8192, "fp8": False},
    ]


def _between(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _pool(rng):
    bits = rng.choice([16, 8, 8, 4, 5, 5])
    return bits, 128 if bits == 16 else rng.choice([32, 64, 128, 128])


def draw(rng):
    kind = rng.choice(["token", "sessions", "ops", "ops", "attn_decode", "attn_prefill",
                       "attn_prefill", "gemm", "gemm", "gemm"])
    bits, group = _pool(rng)
    if kind == "token":
        return {"kind": kind, "layers": rng.randint(1, 8), "context": _between(rng, 16, 65000),
                "bits": bits, "group": group}
    if kind == "sessions":
        return {"kind": kind, "layers": 2, "sessions": rng.randint(2, 16), "bits": bits,
                "fp8": rng.random() < 0.5}
    if kind == "ops":
        tokens = _between(rng, 1, 8192)
        return {"kind": kind, "tokens": tokens, "start": rng.randint(0, MAX_POS - tokens),
                "bits": bits, "group": group}
    if kind == "attn_decode":
        return {"kind": kind, "rows": rng.choice([1, 1, 1, 4, rng.randint(2, 16)]),
                "context": _between(rng, 64, 65000), "bits": bits, "group": group}
    if kind == "attn_prefill":
        tokens = _between(rng, 17, 8192)
        start = rng.choice([0, 0, rng.randint(1, 57344)])
        return {"kind": kind, "tokens": tokens, "start": start, "bits": bits, "group": group}
    proj = rng.choice(["qkv", "o", "gate_up", "down"])
    return {"kind": kind, "proj": proj, "tokens": _between(rng, 1, 8192),
            "fp8": proj != "o" and rng.random() < 0.6}


# -------------------------------------------------------------------- inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def bf16(self, *shape, std=1.0, mean=0.0):
        return (self.normal(*shape, std=std) + mean).to(torch.bfloat16)

    def hidden(self, rows):
        """Residual-stream rows: N(0, 1), 1 % of the channels 20 times larger."""
        x = self.normal(rows, H)
        x[:, torch.randperm(H, generator=self.g, device="cuda")[:H // 100]] *= 20
        return x

    def weight(self, n, k):
        w = torch.randn((n, k), generator=self.g, device="cuda").mul_(W_STD).clamp_(-448, 448)
        return w.to(torch.float8_e4m3fn).view(torch.uint8)

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def arena_rows(self, rows):
        """The arena's rows in a random order of their 16-row pages."""
        p = torch.randperm(rows // 16, generator=self.g, device="cuda").to(torch.int32)
        return (p[:, None] * 16 + torch.arange(16, device="cuda", dtype=torch.int32)).reshape(-1)


def _table(rows, first=0):
    """The engine's page table: an arena row for each position from `first` on
    that has one, -1 for the others, MAX_POS entries."""
    t = torch.full((MAX_POS,), -1, dtype=torch.int32, device="cuda")
    t[first:first + rows.numel()] = rows
    return t


def _pages(n):
    return (n + 15) // 16 * 16


def _fp8(x):
    """Codes and per-tensor scale (amax / 448) of x."""
    s = (x.abs().max() / 448).reshape(1)
    return (x / s).to(torch.float8_e4m3fn).view(torch.uint8), s


def _quantise(x, qmax, group):
    """Codes in [-qmax, qmax] (int32) and one scale per `group` of the last dim."""
    xg = x.view(*x.shape[:-1], D // group, group)
    s = xg.abs().amax(-1) / qmax
    c = torch.round(xg / s[..., None]).clamp_(-qmax, qmax).to(torch.int8)
    return c.view(x.shape), s.contiguous()


def _nibbles(u):
    return (u[..., 0::2] & 15) | ((u[..., 1::2] & 15) << 4)


def _pool_of(r, bits, group, stride):
    """One layer's filled pool: cache_k, cache_v (bytes) and their scales."""
    out = []
    for is_k in (True, False):
        x = r.normal(HK, stride, D)
        if bits == 16:
            out.append((x.to(torch.bfloat16).view(torch.uint8), None))
            continue
        qmax = 127 if bits == 8 else 15 if bits == 5 and is_k else 7
        c, s = _quantise(x, qmax, group)
        del x
        if bits == 8:
            rows = c.view(torch.uint8)
        else:
            u = (c + (qmax + 1)).view(torch.uint8)
            rows = _nibbles(u)
            if qmax == 15:
                b = (u >> 4).view(HK, stride, 16, 8)
                plane = b[..., 0].clone()
                for i in range(1, 8):
                    plane |= b[..., i] << i
                rows = torch.cat([rows, plane], -1)
        out.append((rows.contiguous(), s))
    return out[0][0], out[1][0], out[0][1], out[1][1]


def _values(rows, scale, bits, is_k):
    """The 64-bit values of pool rows [..., row bytes] with scales [..., groups]."""
    if bits == 16:
        return rows.contiguous().view(torch.bfloat16).double()
    if bits == 8:
        c = rows.contiguous().view(torch.int8).double()
    else:
        n = rows[..., :D // 2]
        c = torch.stack([n & 15, n >> 4], -1).flatten(-2).to(torch.int32)
        if bits == 5 and is_k:
            p = rows[..., D // 2:].to(torch.int32)
            c |= torch.stack([((p >> i) & 1) << 4 for i in range(8)], -1).flatten(-2)
            c -= 16
        else:
            c -= 8
        c = c.double()
    s = scale.double().repeat_interleave(D // scale.shape[-1], -1)
    return c * s


def _kv_row_bytes(bits, group):
    kb, vb = {16: (256, 256), 8: (128, 128), 4: (64, 64), 5: (80, 64)}[bits]
    return kb + vb + (0 if bits == 16 else 2 * 4 * (D // group))


# The scales of a model whose projections give values of about 1 (q: 16, so
# that with the 1 / 128 attention scale the logits spread by a few units).
def _layer(r, bits, group, stride):
    wqkv, wgu = r.weight(NQ + 2 * NK, H), r.weight(2 * INTER, H)
    s = 1 / (W_STD * math.sqrt(H))
    ly = {"attn_norm": r.bf16(H, std=0.1, mean=1.0), "ffn_norm": r.bf16(H, std=0.1, mean=1.0),
          "wq": wqkv[:NQ], "wk": wqkv[NQ:NQ + NK], "wv": wqkv[NQ + NK:], "wo": r.weight(H, NQ),
          "wg": wgu[:INTER], "wu": wgu[INTER:], "wd": r.weight(H, INTER), "sq": 16 * s, "sk": s,
          "sv": s, "so": 4 * s, "sg": s, "su": s, "sd": 1 / (W_STD * math.sqrt(INTER))}
    ly["cache_k"], ly["cache_v"], ly["k_scale"], ly["v_scale"] = _pool_of(r, bits, group, stride)
    return ly


def _inputs(case, seed):
    """Everything that is made from the seed, as a dict of tensors."""
    r = _Rand(seed)
    kind = case["kind"]
    if kind in ("token", "sessions"):
        n = case.get("sessions", 1)
        bits, group = case["bits"], case.get("group", 128)
        pos = ([case["context"] - 1] if kind == "token" else
               [int(p) for p in r.ints(MAX_POS, n).tolist()])
        # every session's pages lie in one pool, in random order
        need = [_pages(p + 1) for p in pos]
        stride = _pages(sum(need))
        if kind == "sessions":
            stride = max(stride, MAX_POS)  # the batched step's pool holds a longest sequence
        rows = r.arena_rows(stride)
        pts, at = [], 0
        for k in need:
            pts.append(_table(rows[at:at + k]))
            at += k
        toks = [r.ints(VOCAB, p + 1) for p in pos]
        return {"pos": pos, "pts": pts, "toks": toks, "stride": stride,
                "emb": r.bf16(VOCAB, H, std=0.05), "final_norm": r.bf16(H, std=0.1, mean=1.0),
                "lm_head": r.weight(VOCAB, H),
                "layers": [_layer(r, bits, group, stride) for _ in range(case["layers"])]}
    if kind == "ops":
        t, p0 = case["tokens"], case["start"]
        # the chunk's pages: a run of fresh ones, the pool no larger than it needs
        stride = _pages(p0 % 16 + t)
        pt = _table(torch.arange(t, device="cuda", dtype=torch.int32) + p0 % 16, p0)
        return {"toks": r.ints(VOCAB, t), "emb": r.bf16(VOCAB, H, std=0.02),
                "res": r.hidden(t).to(torch.bfloat16), "branch": r.bf16(t, H),
                "gamma": r.bf16(H, std=0.1, mean=1.0), "gu": r.bf16(t, 2 * INTER),
                "qkv": r.bf16(t, NQ + 2 * NK), "stride": stride, "pt": pt}
    if kind == "attn_decode":
        stride = _pages(case["context"])
        k, v, ks, vs = _pool_of(r, case["bits"], case["group"], stride)
        return {"q": r.bf16(case["rows"], NQ, std=16), "k": k, "v": v, "ks": ks, "vs": vs,
                "stride": stride, "pt": _table(r.arena_rows(stride))}
    if kind == "attn_prefill":
        stride = _pages(case["start"] + case["tokens"])
        k, v, ks, vs = _pool_of(r, case["bits"], case["group"], stride)
        return {"q": r.bf16(case["tokens"], NQ, std=16), "k": k, "v": v, "ks": ks, "vs": vs,
                "stride": stride, "pt": _table(r.arena_rows(stride))}
    # gemm
    t, proj = case["tokens"], case["proj"]
    n, k = _GEMM[proj]
    if proj == "down":
        a = torch.nn.functional.silu(r.normal(t, k)) * r.normal(t, k)
    elif proj == "o":
        a = r.normal(t, k)
    else:
        a = r.hidden(t)
        a *= torch.rsqrt(a.square().mean(-1, keepdim=True))
    got = {"w": r.weight(n, k)}
    if case["fp8"]:
        got["a"], got["a_scale"] = _fp8(a)
    else:
        got["a"] = a.to(torch.bfloat16)
    if proj in ("o", "down"):
        got["res"] = r.hidden(t).to(torch.bfloat16)
    return got


_GEMM = {"qkv": (NQ + 2 * NK, H), "o": (H, NQ), "gate_up": (2 * INTER, H), "down": (H, INTER)}


def _w_scales(proj):
    s = 1 / (W_STD * math.sqrt(_GEMM[proj][1]))
    return {"qkv": (16 * s, s, 0.5 * s), "gate_up": (s, 1.25 * s, s)}.get(proj, (s, s, s))


# ------------------------------------------------------------------- prepare
def _captured(L, step):
    """step() as one HIP graph, as an engine keeps its decode steps."""
    cap = torch.cuda.Stream()
    cap.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(cap):
        L.use_stream(cap)
        step()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=cap):
            step()
    L.use_stream()
    torch.cuda.synchronize()
    return graph


def prepare(case, seed):
    L = _layerops()
    L.use_stream()
    s = _inputs(case, seed)
    s["case"] = case
    kind, dev, bf = case["kind"], "cuda", torch.bfloat16
    if kind in ("token", "sessions"):
        bits, group, n = case["bits"], case.get("group", 128), case.get("sessions", 1)
        s["cos"], s["sin"] = L.rope_tables(THETA, D, MAX_POS)
        kw = dict(eps=EPS, emb_mult=EMB_MULT, resid_mult=RESID, attn_scale=ATTN_SCALE,
                  final_norm=s["final_norm"], lm_head=s["lm_head"], lm_scale=1 / (W_STD * 64),
                  kv_bits=bits, kv_group=group, kv_stride=s["stride"])
        s["hidden"] = torch.empty((n, H), dtype=bf, device=dev)
        s["logits"] = torch.empty((n, VOCAB), dtype=bf, device=dev)
        dims = (s["layers"], H, INTER, HQ, HK, VOCAB, s["emb"], s["cos"], s["sin"])
        if kind == "token":
            s["step"] = L.DecodeStep(*dims, **kw)
            s["d_pos"] = torch.tensor(s["pos"], dtype=torch.int32, device=dev)

            def step():
                s["step"](s["toks"][0], s["d_pos"], s["pts"][0], s["hidden"], s["logits"])
        else:
            s["step"] = L.LayerSteps(*dims, n, **kw)
            m = L.multi_rows_struct()()
            m.n = n
            for i in range(n):
                m.pos[i] = s["pos"][i]
                m.pt[i] = s["pts"][i].data_ptr()
                m.tok[i] = s["toks"][i].data_ptr()
            s["rows"] = torch.from_numpy(np.frombuffer(bytes(m), np.uint8).copy()).to(dev)
            ops = L.OPS_FP8 if case["fp8"] else L.OPS_BF16

            def step():
                s["step"].multi(s["rows"], n, ops, s["hidden"], s["logits"])
        s["graph"] = _captured(L, step)
    elif kind == "ops":
        t = case["tokens"]
        s["cos"], s["sin"] = L.rope_tables(THETA, D, MAX_POS)
        s["work"] = L.fp8_workspace(t)
        s["arena"] = L.KvArena(case["bits"], HK, s["stride"], group=case["group"])
        s["x"] = torch.empty((t, H), dtype=bf, device=dev)
        s["res_out"] = torch.empty((t, H), dtype=bf, device=dev)
        s["codes"] = torch.empty((t, H), dtype=torch.uint8, device=dev)
        s["act_codes"] = torch.empty((t, INTER), dtype=torch.uint8, device=dev)
        s["scales"] = torch.zeros(2, dtype=torch.float32, device=dev)
        s["q_rot"] = torch.empty((t, NQ), dtype=bf, device=dev)
        if t <= 1024:  # decode batches and short prompts are replayed as a graph
            s["graph"] = _captured(L, lambda: _layer_ops(L, s))
    elif kind in ("attn_decode", "attn_prefill"):
        s["out"] = torch.empty_like(s["q"])
        if kind == "attn_decode":
            s["d_pos"] = torch.tensor([case["context"] - case["rows"]], dtype=torch.int32,
                                      device=dev)
            nbytes = L.call_size("granite4_attn_split_scratch_bytes", HQ, case["rows"],
                                 s["stride"])
            s["scratch"] = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    else:
        t, (n, _) = case["tokens"], _GEMM[case["proj"]]
        if case["proj"] == "gate_up":
            s["act"] = torch.empty((t, INTER), dtype=bf, device=dev)
            if case["fp8"]:
                s["work"] = L.fp8_workspace(t)
            else:
                s["gu"] = torch.empty((t, 2 * INTER), dtype=torch.float32, device=dev)
        else:
            s["out"] = torch.empty((t, n), dtype=bf, device=dev)
    return s


# ----------------------------------------------------------------------- run
def _layer_ops(L, s):
    """The embedding, and one layer's ops between its GEMMs."""
    t, p0 = s["case"]["tokens"], s["case"]["start"]
    L.call("granite4_embed_rows", s["toks"], t, s["emb"], VOCAB, H, EMB_MULT, s["x"])
    L.add_rmsnorm_fp8(s["res"], s["branch"], s["gamma"], EPS, s["work"], RESID, s["res_out"],
                      s["codes"], s["scales"][:1])
    L.swiglu_fp8(s["gu"], s["work"], s["act_codes"], s["scales"][1:])
    q, k, v = s["qkv"][:, :NQ], s["qkv"][:, NQ:NQ + NK], s["qkv"][:, NQ + NK:]
    L.rope_append(s["arena"], q, k, v, s["cos"], s["sin"], p0, d_pt=s["pt"], q_rot=s["q_rot"])


def run(s):
    L, case = _layerops(), s["case"]
    kind = case["kind"]
    if kind in ("token", "sessions"):
        s["graph"].replay()
        return {"hidden": s["hidden"], "logits": s["logits"]}
    if kind == "ops":
        if "graph" in s:
            s["graph"].replay()
        else:
            _layer_ops(L, s)
        a = s["arena"]
        return {"embed": s["x"], "res": s["res_out"],
                "normed": s["codes"].view(torch.float8_e4m3fn),
                "act": s["act_codes"].view(torch.float8_e4m3fn), "scales": s["scales"],
                "q": s["q_rot"], "k": a.k, "v": a.v, "k_scale": a.k_scale, "v_scale": a.v_scale}
    if kind == "attn_decode":
        L.call("granite4_attn_paged", s["q"], case["rows"], HQ, HK, D, ATTN_SCALE, s["k"], s["v"],
               s["ks"], s["vs"], case["bits"], case["group"], s["stride"], 0, s["d_pos"], s["pt"],
               None, None, 0, 0, s["scratch"], s["out"])
        return s["out"]
    if kind == "attn_prefill":
        L.call("granite4_prefill_attn", s["q"], case["tokens"], HQ, HK, D, ATTN_SCALE, s["k"],
               s["v"], s["ks"], s["vs"], case["bits"], case["group"], s["stride"], case["start"],
               s["pt"], 0, s["out"])
        return s["out"]
    proj, sc = case["proj"], _w_scales(case["proj"])
    if proj == "gate_up":
        if case["fp8"]:
            act, codes, scale = L.gemm_fp8_swiglu(s["a"], s["a_scale"], s["w"], sc[0], sc[1],
                                                  s["work"], s["act"])
            return {"act": act, "codes": codes.view(torch.float8_e4m3fn), "scale": scale}
        gu = s["gu"]
        L.prefill_gemm(s["a"], s["w"][:INTER], L.GEMM_F32, (sc[0],) * 3, out=gu[:, :INTER])
        L.prefill_gemm(s["a"], s["w"][INTER:], L.GEMM_F32, (sc[1],) * 3, out=gu[:, INTER:])
        return {"gate_up": gu, "act": L.prefill_silu_mul(gu, INTER, case["tokens"], s["act"])}
    kind_out, segs, res = L.GEMM_BF16, (NQ, NQ + NK), None
    if proj != "qkv":
        kind_out, segs, res = L.GEMM_RESIDUAL, None, s["res"]
    if case["fp8"]:
        return L.gemm_fp8(s["a"], s["a_scale"], s["w"], kind_out, sc, segs, s["out"], res, RESID)
    return L.prefill_gemm(s["a"], s["w"], kind_out, sc, segs, s["out"], res, RESID)


# ---------------------------------------------------------------------- work
def _attn_work(rows_pos, rows, kv_positions, bits, group):
    """rows_pos: (query row, position) pairs counted; kv_positions: positions read."""
    return {"bytes": kv_positions * (HK * _kv_row_bytes(bits, group) + 4) + 2 * rows * NQ * 2,
            "flops": 4 * NQ * rows_pos}


def work(case):
    kind = case["kind"]
    if kind in ("token", "sessions"):
        n, bits, group = case.get("sessions", 1), case["bits"], case.get("group", 128)
        weights = (NQ + 2 * NK) * H + H * NQ + 3 * INTER * H
        ctx = case["context"] if kind == "token" else n * MAX_POS // 2
        att = _attn_work(ctx, n, ctx, bits, group)
        return {"bytes": case["layers"] * (weights + att["bytes"]) + VOCAB * H + 2 * n * VOCAB,
                "flops": case["layers"] * (2 * n * weights + att["flops"]) + 2 * n * VOCAB * H}
    if kind == "ops":
        t = case["tokens"]
        rope = 2 * (NQ + 2 * NK) + 2 * NQ + HK * _kv_row_bytes(case["bits"], case["group"]) + 4 + 512
        return {"bytes": t * (4 * H + 4 + 7 * H + 5 * INTER + rope) + 2 * H, "flops": 0}
    if kind == "attn_decode":
        c, r = case["context"], case["rows"]
        return _attn_work(r * c - r * (r - 1) // 2, r, c, case["bits"], case["group"])
    if kind == "attn_prefill":
        t, p0 = case["tokens"], case["start"]
        return _attn_work(t * p0 + t * (t + 1) // 2, t, p0 + t, case["bits"], case["group"])
    t, (n, k) = case["tokens"], _GEMM[case["proj"]]
    moved = n * k + t * k * (1 if case["fp8"] else 2)
    if case["proj"] == "gate_up":
        moved += t * INTER * (3 if case["fp8"] else 10)
    else:
        moved += t * n * (2 if case["proj"] == "qkv" else 4)
    return {"bytes": moved, "flops": 2 * t * n * k}


# ----------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    if kind in ("token", "sessions"):
        # a rounding of one bf16 (or FP8) value travels through the layers
        return {"rel": 0.03 if case.get("fp8") else 0.02, "max": 0.5}
    if kind == "ops":
        # bf16 within an ulp and FP8 codes of it; the pool's bytes are whole numbers
        return {"rel": 0.004, "max": 0.15}
    if kind in ("attn_decode", "attn_prefill"):
        # bf16 logits and probabilities, against ones that are kept in 32 bits
        return {"rel": 0.025, "max": 0.25}
    if case["proj"] == "gate_up" and case["fp8"]:
        # the scale follows one element's bf16 rounding, the codes follow the scale
        return {"rel": 0.02, "max": 0.2}
    return {"rel": 0.003, "max": 0.03}


# --------------------------------------------------------------------- exact
def _norm(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.double()


def _rope(x, pos):
    """x [rows, heads, D], pos [rows]: halves rotated by pos * theta^(-2 i / D)."""
    i = torch.arange(D // 2, device="cuda", dtype=torch.float64)
    ang = pos.double()[:, None, None] * torch.pow(torch.tensor(THETA, dtype=torch.float64,
                                                               device="cuda"), -2 * i / D)
    c, s, a, b = torch.cos(ang), torch.sin(ang), x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _w64(w):
    return w.view(torch.float8_e4m3fn).double()


def _mm(a, w, scale):
    """a [rows, K] . w^T in column blocks."""
    return torch.cat([a @ _w64(w[i:i + 16384]).t() for i in range(0, w.shape[0], 16384)], 1) * scale


def _attend(q, k, v, pos):
    """q [rows, HQ, D] at positions pos; k, v [HK, positions, D]."""
    out = torch.empty_like(q)
    key = torch.arange(k.shape[1], device="cuda")
    for r0 in range(0, q.shape[0], 512):
        p = pos[r0:r0 + 512]
        n = int(p.max()) + 1
        unseen = (key[None, :n] > p[:, None]).repeat_interleave(HQ // HK, 0)
        for h in range(HK):
            g = slice(h * (HQ // HK), (h + 1) * (HQ // HK))
            qq = q[r0:r0 + 512, g].reshape(-1, D)
            e = (qq @ k[h, :n].t()).mul_(ATTN_SCALE).masked_fill_(unseen, -math.inf)
            out[r0:r0 + 512, g] = (torch.softmax(e, -1) @ v[h, :n]).view(-1, HQ // HK, D)
    return out


def _exact_model(case, i):
    bits, n = case["bits"], len(i["pos"])
    pos = torch.tensor(i["pos"], device="cuda")
    x = EMB_MULT * torch.stack([i["emb"][int(i["toks"][r][i["pos"][r]])].double()
                                for r in range(n)])
    for ly in i["layers"]:
        a = _norm(x, ly["attn_norm"])
        q = _rope(_mm(a, ly["wq"], ly["sq"]).view(n, HQ, D), pos)
        k = _rope(_mm(a, ly["wk"], ly["sk"]).view(n, HK, D), pos)
        v = _mm(a, ly["wv"], ly["sv"]).view(n, HK, D)
        o = torch.empty_like(q)
        for r in range(n):
            p = i["pos"][r]
            at = i["pts"][r][:p].long()
            kk, vv = (torch.cat([_values(ly["cache_" + c][:, at], None if bits == 16 else
                                         ly[c + "_scale"][:, at], bits, c == "k"),
                                 new[r][:, None]], 1) for c, new in (("k", k), ("v", v)))
            o[r:r + 1] = _attend(q[r:r + 1], kk, vv, pos[r:r + 1])
            del kk, vv
        x = x + RESID * _mm(o.reshape(n, NQ), ly["wo"], ly["so"])
        a = _norm(x, ly["ffn_norm"])
        act = torch.nn.functional.silu(_mm(a, ly["wg"], ly["sg"])) * _mm(a, ly["wu"], ly["su"])
        x = x + RESID * _mm(act, ly["wd"], ly["sd"])
    hidden = _norm(x, i["final_norm"])
    return {"hidden": hidden, "logits": _mm(hidden, i["lm_head"], 1 / (W_STD * 64))}


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    if kind in ("token", "sessions"):
        return _exact_model(case, i)
    if kind == "ops":
        t, p0 = case["tokens"], case["start"]
        res = i["res"].double() + RESID * i["branch"].double()
        normed = _norm(res, i["gamma"])
        act = torch.nn.functional.silu(i["gu"][:, :INTER].double()) * i["gu"][:, INTER:].double()
        scales = torch.stack([normed.abs().max(), act.abs().max()]) / 448
        pos = torch.arange(p0, p0 + t, device="cuda")
        q = _rope(i["qkv"][:, :NQ].double().view(t, HQ, D), pos)
        return {"embed": EMB_MULT * i["emb"][i["toks"].long()].double(), "res": res,
                "normed": normed / scales[0], "act": act / scales[1], "scales": scales,
                "q": q.reshape(t, NQ), "k": None, "v": None, "k_scale": None, "v_scale": None}
    if kind in ("attn_decode", "attn_prefill"):
        rows = i["q"].shape[0]
        p0 = case["start"] if kind == "attn_prefill" else case["context"] - rows
        at = i["pt"][:p0 + rows].long()
        k, v = (_values(i[c][:, at], None if case["bits"] == 16 else i[c + "s"][:, at],
                        case["bits"], c == "k") for c in ("k", "v"))
        pos = torch.arange(p0, p0 + rows, device="cuda")
        return _attend(i["q"].double().view(rows, HQ, D), k, v, pos).reshape(rows, NQ)
    proj, sc = case["proj"], _w_scales(case["proj"])
    a = _w64(i["a"]) * i["a_scale"].double() if case["fp8"] else i["a"].double()
    y = _mm(a, i["w"], 1.0)
    if proj == "gate_up":
        y[:, :INTER] *= sc[0]
        y[:, INTER:] *= sc[1]
        act = torch.nn.functional.silu(y[:, :INTER]) * y[:, INTER:]
        if not case["fp8"]:
            return {"gate_up": y, "act": act}
        scale = act.abs().max().reshape(1) / 448
        return {"act": act, "codes": act / scale, "scale": scale}
    if proj == "qkv":
        y[:, :NQ] *= sc[0]
        y[:, NQ:NQ + NK] *= sc[1]
        y[:, NQ + NK:] *= sc[2]
        return y
    return i["res"].double() + RESID * sc[0] * y
