"""The work that is timed: the expert's Euler loop and the kernels that surround it in one policy call.

A policy step makes the modulation rows of every Euler step (``StepModulations``), projects the VLM context onto
each layer's cross-attention caches (``SourcePrepare``), integrates the action chunk (``ExpertMegakernel.run``,
``run_first``, ``run_all``) and appends the call's register rows to the register memory (``mkx_ring_append``).
The sizes are those of the named workloads in ``mkx.synthetic``; ``draw`` spreads them over what the library takes:
widths 256, 768 and 1024, 2 to 16 layers, 1 to 8 samples, 1 to 50 action rows, with and without register rows, 16 to
256 memory rows, 1 to 1024 source rows (ragged over the samples too), bf16 and fp8 weights, 1 to 10 steps.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "reki-megakernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HD, A, EPS, TDIM = 64, 32, 1e-6, 256

# One expert and one call of it. op: run = Euler steps 2..N from x after step 1; all = steps 1..N in one launch, with
# the register rows' K/V; first = step 1 alone with the register rows' K/V; mods, source, ring = the kernels around.
# T action rows and R register rows (loop: they ride in every step); PM memory rows of which the first kv are
# not filled yet; S valid of SP source rows (ragged: the samples' S and kv differ); C = context width.
_BASE = {"op": "run", "L": 10, "H": 768, "I": 3072, "fp8": False, "gelu": False, "B": 1, "T": 10, "R": 32, "loop": True,
         "PM": 96, "kv": 0, "S": 300, "SP": 300, "C": 2048, "steps": 10, "adim": 7, "ragged": False}
_WIDE = {"L": 16, "H": 1024, "I": 4096, "fp8": True, "T": 50}


def _case(name, **kw):
    return {"name": name, **_BASE, **kw}


def listed():
    return [
        # the modulation rows of one robot's call, and of eight batched calls: the smallest launches of a call
        _case("mods_b1", op="mods"),
        _case("mods_b8", op="mods", B=8),
        # the register memory of eight streams after a call
        _case("ring_b8", op="ring", B=8),
        # source caches of one call, and of eight whose prompts have different lengths
        _case("source_b1", op="source"),
        _case("source_b8", op="source", B=8, ragged=True),
        # step 1 of a split call (its register rows' K/V go to the ring): the shortest Euler launch
        _case("first_b1", op="first", steps=1),
        # the headline: steps 2-10 of one robot's chunk with the register rows in every step
        _case("run_b1"),
        # the same in the ten-row layout: register rows only in step 1, the memory not full yet, a short prompt
        _case("run_b1_rows10", loop=False, kv=32, S=182, SP=256),
        # a long prompt and eight frames of register memory
        _case("run_b1_long", S=1024, SP=1024, PM=256),
        # eight independent chunks (batched evaluation, several robots), steps 1-10 in one launch
        _case("all_b8", op="all", B=8),
        # the wide fp8 expert with fifty-action chunks, for one robot and for four
        _case("run_fp8_b1", **_WIDE),
        _case("run_fp8_b4", B=4, **_WIDE),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    most = work(_case("most", B=4, **_WIDE))["flops"]
    while True:
        op = rng.choice(["run"] * 8 + ["all"] * 4 + ["first"] * 3 + ["mods"] * 3 + ["source"] * 3 + ["ring"] * 3)
        H, I, Lmax, Bmax = rng.choice([(768, 3072, 10, 8)] * 3 + [(1024, 4096, 16, 6)] * 2 + [(256, 512, 4, 8)])
        R = rng.choice([0, 3, 16, 32, 32, 32])
        if op in ("ring", "first"):
            R = max(R, 1)
        T = _log_int(rng, 1, 50)
        PM = rng.choice([_log_int(rng, max(16, R), 256), 96, 32 * rng.randint(1, 8)])
        SP = _log_int(rng, 8, 1024)
        S = rng.choice([SP, rng.randint(max(1, SP // 2), SP)])
        C = rng.choice([2048, 2048, 960, 96])
        c = {"op": op, "L": rng.randint(2, Lmax), "H": H, "I": I, "fp8": rng.random() < 0.4, "gelu": rng.random() < 0.3,
             "B": _log_int(rng, 1, Bmax), "T": T, "R": R, "loop": op == "all" or rng.random() < 0.7, "PM": PM,
             "kv": rng.choice([0, 0, rng.randint(0, PM - 1)]), "S": S, "SP": SP, "C": C,
             "steps": 1 if op == "first" else rng.randint(2, 10), "adim": rng.choice([7, 7, 14, rng.randint(1, 24)]),
             "ragged": rng.random() < 0.4}
        rows = -(-(c["T"] + c["R"]) // 16) * 16 * c["B"]
        if rows <= 384 and c["B"] * c["T"] <= 200 and c["adim"] * H <= 16384 and work(c)["flops"] <= most:
            return c


def _lens(c):
    """(ca_len, kv_start) of each sample."""
    if not c["ragged"]:
        return [c["S"]] * c["B"], [c["kv"]] * c["B"]
    return ([max(1, c["S"] - (37 * b) % max(1, c["S"])) for b in range(c["B"])],
            [(c["kv"] + 32 * b) % c["PM"] for b in range(c["B"])])


def _modw(c):
    return 9 * c["L"] * c["H"] + 2 * c["H"]


def _m_q(c, first=False):
    return c["T"] + (c["R"] if c["loop"] or first else 0)


def work(case):
    c = case
    L, H, I, B, N = c["L"], c["H"], c["I"], c["B"], c["steps"]
    lens, kvs = _lens(c)
    if c["op"] == "mods":
        rows, n = B * N, _modw(c)
        return {"bytes": 2 * (n * H + H * H + H * TDIM) + 4 * (n + 2 * H + B * H + rows * n),
                "flops": 2 * rows * n * H + 2 * N * H * (H + TDIM)}
    if c["op"] == "source":
        out = 2 * L * B * c["SP"] * H * 2
        return {"bytes": 2 * L * H * c["C"] * 2 + B * c["SP"] * c["C"] * 2 + out, "flops": 4 * sum(lens) * c["C"] * H * L}
    if c["op"] == "ring":
        return {"bytes": 2 * 2 * L * B * c["PM"] * H * 2, "flops": 3 * L * B * c["PM"] * H}
    steps = N - 1 if c["op"] == "run" else N
    mq = _m_q(c, c["op"] != "run")
    keys = sum(c["PM"] - k + mq + s for k, s in zip(kvs, lens))
    w = L * (6 * H * H + 3 * H * I) * (1 if c["fp8"] else 2)
    kv = 2 * 2 * L * H * sum(c["PM"] - k + s for k, s in zip(kvs, lens))
    # every weight and cache is read once in each step: together they do not stay on the chip between steps
    return {"bytes": steps * (w + kv + 4 * B * _modw(c) + 8 * A * H),
            "flops": steps * (2 * B * mq * L * (6 * H * H + 3 * H * I) + 4 * L * H * mq * keys)}


# About four times the errors seen against 64-bit results over the listed cases and 24 drawn ones (2-norm; largest
# difference): mods 2.5e-6 / 1.3e-5, source 2.9e-3 / 2.9e-2 (bf16 results of bf16 products), the Euler steps 3.1e-4 /
# 2.2e-3 (fp16 operands through up to 16 layers and 10 steps), the register rows' K/V 1.9e-3 / 7.8e-3 (bf16 results).
# Two correct implementations differ by up to about that much each. The ring's rounding order is part of its interface.
_TOL = {
    "mods": {"rel": 1e-5, "max": 5e-5},
    "source": {"rel": 1.2e-2, "max": 1.2e-1},
    "run": {"rel": 1.2e-3, "max": 9e-3},
    "kv": {"rel": 8e-3, "max": 3e-2},
}


def tolerance(case):
    if case["op"] == "ring":
        return "exact"
    if case["op"] in ("mods", "source", "run"):
        return dict(_TOL[case["op"]])
    return dict(_TOL["kv"])  # x in fp32 and the register rows' K/V in bf16


# ------------------------------------------------------------------------------------------------ inputs


def _dev():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


class _Gen:
    def __init__(self, seed):
        self.dev = _dev()
        self.g = torch.Generator(device=self.dev).manual_seed(1000003 * int(seed) + 17)

    def __call__(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=self.dev) * std


def _rope(n, start=0):
    """(cos, sin) [n, 64] fp32 of rotate-half RoPE at positions start..start+n-1."""
    f = (torch.arange(n, dtype=torch.float64) + start)[:, None] * 10000.0 ** (-torch.arange(0, HD, 2, dtype=torch.float64) / HD)
    f = torch.cat([f, f], -1)
    return torch.cos(f).float().to(_dev()), torch.sin(f).float().to(_dev())


def _cache(g, c, rows, v_std, valid):
    """One layer's (K, V) [B, rows, NH, 64] bf16: K a normed and rotated head row, V a projection; other rows zero."""
    shape = (c["B"], rows, c["H"] // HD, HD)
    k = g(*shape)
    k = k * torch.rsqrt((k * k).mean(-1, keepdim=True)) * (1 + g(HD, std=0.02))
    return (k * valid).to(torch.bfloat16), (g(*shape, std=v_std) * valid).to(torch.bfloat16)


def _linear(g, c, *shape):
    """Weights N(0, 0.02): (bf16, None), or e4m3 codes with a scale per output channel (largest magnitude = 448)."""
    w = g(*shape, std=0.02)
    if not c["fp8"]:
        return w.to(torch.bfloat16), None
    s = w.abs().amax(-1) / 448.0
    return (w / s[..., None]).to(torch.float8_e4m3fn), s


def _expert(c, seed):
    """Weights, caches and inputs of an Euler launch, as plain tensors."""
    g = _Gen(seed)
    L, H, I, B = c["L"], c["H"], c["I"], c["B"]
    NH = H // HD
    w = {}
    for name, n, k in (("wqkv", 3 * H, H), ("wo", H, H), ("wqca", H, H), ("woca", H, H), ("wg", I, H), ("wu", I, H), ("wd", H, I)):
        parts = [_linear(g, c, n, k) for _ in range(L)]
        w[name] = torch.stack([p[0] for p in parts])
        if c["fp8"]:
            w[name + "_scale"] = torch.stack([p[1] for p in parts])
    for name in ("qn", "kn", "qcan"):
        w[name] = g(L, HD, std=0.02).to(torch.bfloat16)
    for name, shape in (("win", (A, H)), ("bin", (H,)), ("wout", (A, H)), ("bout", (A,))):
        w[name] = g(*shape, std=0.02).to(torch.bfloat16).float()
    if c["R"] > 0:
        w["reg_tok"] = g(c["R"], H, std=0.02).to(torch.bfloat16)
    lens, kvs = _lens(c)
    dev = g.dev
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    at = lambda n: torch.arange(n, device=dev)[None, :]  # noqa: E731
    src_ok = (at(c["SP"]) < i32(lens)[:, None])[:, :, None, None]
    mem_ok = (at(c["PM"]) >= i32(kvs)[:, None])[:, :, None, None]
    mem = [_cache(g, c, c["PM"], 0.02 * math.sqrt(H), mem_ok) for _ in range(L)]
    src = [_cache(g, c, c["SP"], 0.02 * math.sqrt(c["C"]), src_ok) for _ in range(L)]
    mq, mf = _m_q(c), c["T"] + c["R"]
    x = g(B, c["T"], A)
    if c["op"] == "run":
        x[..., c["adim"]:] *= 0.02  # after step 1 the padded dims hold dt v only
    mods = g(B, c["steps"], _modw(c), std=0.33)  # silu(c) W^T of c ~ N(0, 1): see StepModulations
    return {"w": w, "mem": mem, "src": src, "kvs": i32(kvs), "lens": i32(lens), "sa": _rope(mq, c["PM"]), "ca": _rope(mq),
            "sa1": _rope(mf, c["PM"]), "ca1": _rope(mf), "x": x, "mods": mods,
            "dt": torch.full((1,), -1.0 / max(c["steps"], 10 if c["op"] == "first" else 1), device=dev), "NH": NH}


def _mods_inputs(c, seed):
    g = _Gen(seed)
    H = c["H"]
    bf = torch.bfloat16
    return ([g(H, TDIM, std=0.02).to(bf), g(H, std=0.02).to(bf), g(H, H, std=0.02).to(bf), g(H, std=0.02).to(bf),
             g(_modw(c), H, std=0.02).to(bf), g(_modw(c), std=0.02).to(bf)], g(c["B"], H))


def _source_inputs(c, seed):
    g = _Gen(seed)
    bf = torch.bfloat16
    layers = [(g(c["H"], c["C"], std=0.02).to(bf), g(c["H"], c["C"], std=0.02).to(bf), g(HD, std=0.02).to(bf)) for _ in range(c["L"])]
    ctx = g(c["B"], c["SP"], c["C"]).to(bf)
    lens = torch.tensor(_lens(c)[0], dtype=torch.int32, device=g.dev)
    ctx *= (torch.arange(c["SP"], device=g.dev)[None, :] < lens[:, None])[:, :, None]
    return layers, ctx, lens


def _ring_inputs(c, seed):
    g = _Gen(seed)
    L, B, PM, NH, R = c["L"], c["B"], c["PM"], c["H"] // HD, c["R"]
    kvs = torch.tensor(_lens(c)[1], dtype=torch.int32, device=g.dev)
    ok = (torch.arange(PM, device=g.dev)[None, :] >= kvs[:, None])[:, :, None, None]
    mem = [_cache(g, c, PM, 0.02 * math.sqrt(c["H"]), ok) for _ in range(L)]
    ck = g(L, B, R, NH, HD).to(torch.bfloat16)
    cv = g(L, B, R, NH, HD, std=0.55).to(torch.bfloat16)
    turn = []
    for delta in (-R, -(c["T"] + R)):  # kept rows move up by R, appended rows from their place in the call
        f = 10000.0 ** (-torch.arange(0, HD, 2, dtype=torch.float64) / HD) * delta
        f = torch.cat([f, f])
        turn.append((torch.cos(f).float().to(g.dev), torch.sin(f).float().to(g.dev)))
    return mem, ck, cv, kvs, turn


class _Bag:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    c = case
    if c["op"] == "mods":
        from mkx.modulations import StepModulations
        w, sc = _mods_inputs(c, seed)
        return {"op": "mods", "step": StepModulations(*w), "n": c["steps"], "sc": sc}
    if c["op"] == "source":
        from mkx.prepare import SourcePrepare
        layers, ctx, lens = _source_inputs(c, seed)
        NH = c["H"] // HD
        tree = [_Bag(cross_attn=_Bag(n_kv_heads=NH, head_dim=HD, k_proj=_Bag(weight=k), v_proj=_Bag(weight=v),
                                     k_norm=_Bag(weight=n, eps=EPS))) for k, v, n in layers]
        model = _Bag(vlm_with_expert=_Bag(action_expert=_Bag(layers=tree)))
        return {"op": "source", "prep": SourcePrepare(model), "ctx": ctx, "lens": lens}
    if c["op"] == "ring":
        from mkx import _lib
        mem, ck, cv, kvs, turn = _ring_inputs(c, seed)
        out = [(torch.empty_like(k), torch.empty_like(v)) for k, v in mem]
        kv_out = torch.empty_like(kvs)
        a = _lib.MkxRingArgs(L=c["L"], B=c["B"], NH=c["H"] // HD, HD=HD, PM=c["PM"], R=c["R"])
        a.cur_k, a.cur_v = ck.data_ptr(), cv.data_ptr()
        for l in range(c["L"]):
            a.memk_in[l], a.memv_in[l] = mem[l][0].data_ptr(), mem[l][1].data_ptr()
            a.memk_out[l], a.memv_out[l] = out[l][0].data_ptr(), out[l][1].data_ptr()
        a.mem_stride_b = c["PM"] * c["H"]
        a.kv_start_in, a.kv_start_out = kvs.data_ptr(), kv_out.data_ptr()
        a.shift_cos, a.shift_sin = turn[0][0].data_ptr(), turn[0][1].data_ptr()
        a.new_cos, a.new_sin = turn[1][0].data_ptr(), turn[1][1].data_ptr()
        return {"op": "ring", "lib": _lib, "args": a, "out": out, "kv": kv_out, "keep": (mem, ck, cv, kvs, turn)}
    from mkx import ExpertMegakernel
    from mkx.pack import FORMAT, PackedExpert
    from mkx.synthetic import Past
    e = _expert(c, seed)
    meta = {"format": FORMAT, "L": c["L"], "H": c["H"], "NH": e["NH"], "HD": HD, "I": c["I"], "A": A, "eps": EPS, "qk_eps": EPS,
            "activation": "gelu_tanh" if c["gelu"] else "silu", "weight_dtype": "fp8_e4m3" if c["fp8"] else "bf16"}
    mk = ExpertMegakernel.from_packed(PackedExpert(e["w"], meta))
    one = (lambda t: t[0]) if c["B"] == 1 else (lambda t: t)
    st = {"mem_kv": [(one(k), one(v)) for k, v in e["mem"]], "sa_pe": e["sa"], "ca_pe": e["ca"], "sa_pe_first": e["sa1"],
          "ca_pe_first": e["ca1"], "kv_start": e["kvs"], "ca_len": e["lens"]}
    past = Past(st, [(one(k), one(v)) for k, v in e["src"]])
    return {"op": c["op"], "mk": mk, "x": e["x"], "mods": one(e["mods"]), "dt": e["dt"], "past": past, "adim": c["adim"]}


def run(state):
    s = state
    if s["op"] == "mods":
        return s["step"](s["n"], s["sc"])
    if s["op"] == "source":
        return s["prep"](s["ctx"], s["lens"])
    if s["op"] == "ring":
        lib = s["lib"]
        lib.check(lib.lib().mkx_ring_append(ctypes.byref(s["args"]), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
                  "mkx_ring_append")
        return s["out"], s["kv"]
    if s["op"] == "run":
        return s["mk"].run(s["x"], s["mods"], s["dt"], s["past"], s["adim"])
    call = s["mk"].run_first if s["op"] == "first" else s["mk"].run_all
    return call(s["x"], s["mods"], s["dt"], s["past"], s["adim"])


# ------------------------------------------------------------------------------------------------ 64-bit results


def _rot(x, cos, sin):
    return x * cos + torch.cat([-x[..., HD // 2:], x[..., : HD // 2]], -1) * sin


def _norm(x, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, ok):
    """q [B, M, NH, 64], k / v [B, N, NH, 64], ok [B, N] valid keys."""
    s = torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) / math.sqrt(HD)
    s = s.masked_fill(~ok[:, None, None, :], -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.transpose(1, 2).contiguous()).transpose(1, 2)


def _exact_steps(c, seed):
    e = _expert(c, seed)
    d = torch.float64
    B, T, H, L, NH = c["B"], c["T"], c["H"], c["L"], e["NH"]
    first = c["op"] != "run"
    M = _m_q(c, first)
    R = M - T
    sa, ca = (e["sa1"], e["ca1"]) if first else (e["sa"], e["ca"])
    sa, ca = ([t.to(d)[:, None, :] for t in p] for p in (sa, ca))
    dev = e["x"].device

    def lin(name, l):
        w = e["w"][name][l].float().to(d)
        return w * e["w"][name + "_scale"][l].to(d)[:, None] if c["fp8"] else w

    small = {k: e["w"][k].to(d) for k in ("qn", "kn", "qcan", "win", "bin", "wout", "bout")}
    reg = e["w"]["reg_tok"].to(d)[None].expand(B, -1, -1) if R > 0 else None
    mem_ok = torch.arange(c["PM"], device=dev)[None] >= e["kvs"][:, None]
    own_ok = torch.ones(B, M, dtype=torch.bool, device=dev)
    src_ok = torch.arange(c["SP"], device=dev)[None] < e["lens"][:, None]
    names = ("wqkv", "wo", "wqca", "woca", "wg", "wu", "wd")
    weights = [{n: lin(n, l) for n in names} for l in range(L)]
    x, dt = e["x"].to(d), e["dt"].to(d)
    act = (lambda t: F.gelu(t, approximate="tanh")) if c["gelu"] else F.silu
    keep_k, keep_v = [], []
    lead = torch.arange(A, device=dev) < c["adim"]
    row0 = 1 if c["op"] == "run" else 0
    for s in range(row0, c["steps"]):
        m = e["mods"][:, s].to(d)
        x = torch.where(lead, x, torch.zeros_like(x))
        h = x @ small["win"] + small["bin"]
        if R > 0:
            h = torch.cat([h, reg], 1)
        for l in range(L):
            w = weights[l]
            mod = [t[:, None, :] for t in m[:, 9 * l * H: 9 * (l + 1) * H].split(H, -1)]
            qkv = ((_norm(h) * (1 + mod[0]) + mod[1]) @ w["wqkv"].T).view(B, M, 3, NH, HD)
            q = _rot(_norm(qkv[:, :, 0]) * (1 + small["qn"][l]), *sa)
            k = _rot(_norm(qkv[:, :, 1]) * (1 + small["kn"][l]), *sa)
            v = qkv[:, :, 2]
            if first and s == 0:
                keep_k.append(k[:, T:])
                keep_v.append(v[:, T:])
            y = _attend(q, torch.cat([e["mem"][l][0].to(d), k], 1), torch.cat([e["mem"][l][1].to(d), v], 1),
                        torch.cat([mem_ok, own_ok], 1))
            h = h + (y.reshape(B, M, H) @ w["wo"].T) * mod[2]
            q = ((_norm(h) * (1 + mod[3]) + mod[4]) @ w["wqca"].T).view(B, M, NH, HD)
            q = _rot(_norm(q) * (1 + small["qcan"][l]), *ca)
            y = _attend(q, e["src"][l][0].to(d), e["src"][l][1].to(d), src_ok)
            h = h + (y.reshape(B, M, H) @ w["woca"].T) * mod[5]
            a = _norm(h) * (1 + mod[6]) + mod[7]
            h = h + ((act(a @ w["wg"].T) * (a @ w["wu"].T)) @ w["wd"].T) * mod[8]
        f = m[:, 9 * L * H:].split(H, -1)
        o = _norm(h[:, :T]) * (1 + f[0][:, None]) + f[1][:, None]
        x = x + dt * (o @ small["wout"].T + small["bout"])
    if not first:
        return x
    if R == 0:
        return x, None, None
    return x, torch.stack(keep_k), torch.stack(keep_v)


def exact(case, seed):
    c = case
    d = torch.float64
    if c["op"] == "mods":
        (t1w, t1b, t2w, t2b, mw, mb), sc = _mods_inputs(c, seed)
        t = 1.0 - torch.arange(c["steps"], dtype=d, device=sc.device) / c["steps"]
        f = torch.exp(-math.log(10000.0) * torch.arange(TDIM // 2, dtype=d, device=sc.device) / (TDIM // 2))
        a = 1000.0 * t[:, None] * f[None]
        emb = torch.cat([torch.cos(a), torch.sin(a)], -1)
        z = F.silu(emb @ t1w.to(d).T + t1b.to(d)) @ t2w.to(d).T + t2b.to(d)
        mods = F.silu(z[None] + sc.to(d)[:, None]) @ mw.to(d).T + mb.to(d)
        return (mods[0] if c["B"] == 1 else mods), torch.full((1,), -1.0 / c["steps"], dtype=d, device=sc.device)
    if c["op"] == "source":
        layers, ctx, lens = _source_inputs(c, seed)
        NH = c["H"] // HD
        cos, sin = (t.to(d)[:, None, :] for t in _rope(c["SP"]))
        ok = (torch.arange(c["SP"], device=ctx.device)[None] < lens[:, None])[:, :, None, None]
        x, out = ctx.to(d), []
        for kw, vw, n in layers:
            k = (x @ kw.to(d).T).view(c["B"], c["SP"], NH, HD)
            v = (x @ vw.to(d).T).view(c["B"], c["SP"], NH, HD)
            out.append((_rot(_norm(k) * (1 + n.to(d)), cos, sin) * ok, v * ok))
        return out
    if c["op"] == "ring":
        mem, ck, cv, kvs, turn = _ring_inputs(c, seed)
        R = c["R"]
        kv = torch.clamp(kvs - R, min=0)
        ok = (torch.arange(c["PM"], device=kvs.device)[None] >= kv[:, None])[:, :, None, None]
        turn = [[t.to(d) for t in p] for p in turn]
        out = []
        for l, (k, v) in enumerate(mem):
            k2 = torch.cat([_rot(k[:, R:].to(d), *turn[0]), _rot(ck[l].to(d), *turn[1])], 1)
            out.append((k2 * ok, torch.cat([v[:, R:], cv[l]], 1).to(d) * ok))
        return out, kv
    return _exact_steps(c, seed)
