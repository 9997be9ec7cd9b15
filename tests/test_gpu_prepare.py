"""GPU: ``mkx_prepare_source`` (through the C ABI, via mkx.prepare.SourcePrepare) against the CPU oracle's
``register_prepare`` in ``mirror`` mode (bf16 rounding after the projection, the norm and the rotation,
the points the kernel rounds at), and the expert run on the kernel's caches against the fp32 oracle.

Tolerance: accumulation order (MFMA vs the CPU's) and rsqrt can move a bf16 rounding by one unit, and the
rotation mixes the two halves of a head, so K is bounded per RoPE pair, |delta| <= 2^-6 |(x_d, x_d+32)|,
and V per element, |delta| <= 2^-7 |v| + 2^-12. A wrong position, sign, norm weight or head fails both by
orders of magnitude."""
import ctypes
import json
from dataclasses import replace

import pytest
import torch

from _cases import TINY, diff, make_case, oracle_dims, oracle_steps
from mkx import ExpertMegakernel, _lib, synthetic as SY
from mkx.prepare import SourcePrepare, rope_table
from oracle import expert_ref as ER

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


def _report(name, **kv):
    print(json.dumps({"case": name, **kv}), flush=True)


def _check_prepare(name, cfg, ca_len=None):
    W = SY.make_weights(cfg, 0)
    model = SY.SyntheticReki(cfg, W, device="cuda")
    inp = SY.make_inputs(cfg)
    ca_len = [cfg.S] * cfg.B if ca_len is None else ca_len
    ctx = inp["ctx"]
    prep = SourcePrepare(model)
    kv = prep(ctx.cuda(), ca_len)
    torch.cuda.synchronize()
    ref = ER.register_prepare(ctx, ca_len, inp["mem_states"][:, :0], [0] * cfg.B, SY.oracle_weights(W), oracle_dims(cfg),
                              cfg.m_q, mode="mirror")
    gk = torch.stack([k for k, _ in kv]).float().cpu()  # [L, B, SP, NH, 64]
    gv = torch.stack([v for _, v in kv]).float().cpu()
    rk, rv = ref["kca"].float(), ref["vca"].float()
    pn = torch.sqrt(rk[..., :32] ** 2 + rk[..., 32:] ** 2).repeat(1, 1, 1, 1, 2)
    dk, dv = (gk - rk).abs(), (gv - rv).abs()
    exact_k = float((dk == 0).float().mean())
    exact_v = float((dv == 0).float().mean())
    _report(name, k_max=float(dk.max()), v_max=float(dv.max()), k_exact_frac=exact_k, v_exact_frac=exact_v)
    assert (dk <= 2.0 ** -6 * pn + 1e-6).all()
    assert (dv <= 2.0 ** -7 * rv.abs() + 2.0 ** -12).all()
    for b, n in enumerate(ca_len):
        n = min(max(n, 0), cfg.SP)
        assert (gk[:, b, n:] == 0).all() and (gv[:, b, n:] == 0).all()
    return model, kv


def test_prepare_tiny():
    _check_prepare("prepare tiny (C 96, SP 48)", TINY)


def test_prepare_odd_head_count():
    # three heads: the workgroups take heads in pairs, so the last pair's second head is computed and not stored
    _check_prepare("prepare NH 3 (odd head pair)", replace(TINY, H=192, NH=3, I=384))


def test_prepare_config_A_context():
    _check_prepare("prepare A (L10, C 2048, S 300)", SY.WORKLOADS["A"])


def test_prepare_batch_with_ragged_lengths():
    cfg = replace(SY.WORKLOADS["A"], B=4, L=3)
    _check_prepare("prepare B4 ragged", cfg, ca_len=[300, 1, 0, 150])


def test_prepare_wide_expert():
    cfg = replace(SY.WORKLOADS["D"], L=4)
    _check_prepare("prepare D shape (NH16, 4 layers)", cfg)


@pytest.mark.parametrize("B, SP, C, lens", [
    (1, 5, 32, [5]),                         # one k-block: three of the four waves have none
    (3, 37, 160, [37, 0, 20]),               # an empty sample between others; waves with one and with two k-blocks
    (2, 64, 288, [64, 48]),                  # whole row tiles; nine k-blocks
    (5, 31, 96, [1, 31, 16, 17, 30]),        # samples that end inside, at and past a row tile
    (66, 3, 64, [b % 4 for b in range(66)]),  # more samples than are numbered densely
    (64, 3, 64, [(3 * b) % 4 for b in range(64)]),
    (1, 600, 96, [333]),                     # fewer valid rows than row groups launched
    (4, 300, 4096, [300, 300, 299, 41]),     # more than one block of row groups
    (2, 1024, 2048, [1000, 3]),
])
def test_prepare_numbered_rows(B, SP, C, lens):
    """Valid rows are numbered densely over up to 64 samples and the rows past each sample's length zeroed by the row
    groups' workgroups; k-blocks are dealt over the waves. The tolerance is the module's (one bf16 rounding)."""
    _check_prepare(f"prepare B {B}, SP {SP}, C {C}", replace(TINY, B=B, S=SP, SP=SP, ctx_dim=C), ca_len=lens)


@pytest.mark.parametrize("B", [2, 70])
def test_prepare_clamps_lengths(B):
    """Lengths outside [0, SP] give the same bits as the clamped ones, densely numbered (2 samples) or not (70)."""
    cfg = replace(TINY, B=B, S=33, SP=33)
    prep = SourcePrepare(SY.SyntheticReki(cfg, SY.make_weights(cfg, 0), device="cuda"))
    ctx = SY.make_inputs(cfg)["ctx"].cuda()
    wild = [(-2, 40)[b % 2] for b in range(B)]
    for (k0, v0), (k1, v1) in zip(prep(ctx, wild), prep(ctx, [min(max(n, 0), 33) for n in wild])):
        assert torch.equal(k0, k1) and torch.equal(v0, v1)


def test_expert_on_kernel_prepared_caches():
    """Euler steps 2..N on caches from the kernel: within the tight bound of the fp32 oracle run on the
    same caches, and close to the run on the PyTorch-prepared caches."""
    case = make_case(SY.WORKLOADS["A"])
    cfg, model, past = case["cfg"], case["model"], case["past"]
    x1, _, _ = model._expert_first_step(case["noise"], past, None, case["mods"][..., :1, :], case["dt"], cfg.action_dim)
    mk = ExpertMegakernel(model)
    x_torch = mk.run(x1, case["mods"], case["dt"], past, cfg.action_dim)
    past.cross_attn_kv = SourcePrepare(model)(case["inp"]["ctx"].cuda()[0], [cfg.S])
    x_kern = mk.run(x1, case["mods"], case["dt"], past, cfg.action_dim)
    mk.check()
    torch.cuda.synchronize()
    r32 = oracle_steps(case, x1, 1, cfg.num_steps - 1, "fp32")
    m, a = diff(x_kern, r32, cfg.action_dim)
    mt, _ = diff(x_kern, x_torch, cfg.action_dim)
    _report("expert on kernel caches (A)", vs_fp32_max=m, vs_fp32_mean=a, vs_torch_caches_max=mt)
    assert m <= 1e-3 and a <= 2e-4
    assert mt <= 1e-2


def test_prepare_timing_config_A():
    """Times one preparation of config A's source (10 layers, 300 x 2048 context); reported, not asserted."""
    cfg = SY.WORKLOADS["A"]
    model = SY.SyntheticReki(cfg, SY.make_weights(cfg, 0), device="cuda")
    ctx = SY.make_inputs(cfg)["ctx"].cuda()
    prep = SourcePrepare(model)
    for _ in range(3):
        prep(ctx, [cfg.S])
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(20):
        prep(ctx, [cfg.S])
    e1.record()
    torch.cuda.synchronize()
    us = e0.elapsed_time(e1) * 1e3 / 20
    inp = SY.make_inputs(cfg)
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0.record()
    for _ in range(5):
        model.register_prepare(inp["ctx"], inp["mem_states"])
    t1.record()
    torch.cuda.synchronize()
    _report("prepare timing A", kernel_us=us, torch_register_prepare_us=t0.elapsed_time(t1) * 1e3 / 5)


def test_prepare_rejects_more_rows_than_the_handle_stages():
    from mkx._lib import MkxError
    model = SY.SyntheticReki(TINY, SY.make_weights(TINY, 0), device="cuda")
    prep = SourcePrepare(model, max_rows=TINY.SP - 1)
    with pytest.raises(MkxError):
        prep(SY.make_inputs(TINY)["ctx"].cuda(), [TINY.S])
    prep.close()


def test_whole_call_captured_in_one_graph_replays_match_eager():
    """Step modulations (modulation input and projection), source caches and Euler steps 1..N captured as one
    HIP graph: every replay, with eager work and a synchronisation between replays, equals the eager call bit
    for bit."""
    from mkx.modulations import StepModulations
    case = make_case(SY.WORKLOADS["A"])
    cfg, model, past, W = case["cfg"], case["model"], case["past"], case["W"]
    mk = ExpertMegakernel(model)
    prep = SourcePrepare(model)
    step_mods = StepModulations(*(W[k].cuda() for k in ("t1_w", "t1_b", "t2_w", "t2_b", "mod_w", "mod_b")))
    sc = case["inp"]["state_cond"].cuda()
    ctx = case["inp"]["ctx"].cuda()
    ca_len = torch.tensor([cfg.S], dtype=torch.int32, device="cuda")
    out = {}

    def call():
        mods, dt = step_mods(cfg.num_steps, sc)
        past.cross_attn_kv = [(k[0], v[0]) for k, v in prep(ctx, ca_len)]
        out["x"], out["k"], out["v"] = mk.run_all(case["noise"], mods, dt, past, cfg.action_dim)

    call()
    mk.check()
    torch.cuda.synchronize()
    x_e, k_e = out["x"].clone(), out["k"].clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()  # warm-up on a side stream, as capture requires
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    torch.cuda.synchronize()
    times = []
    for i in range(3):
        out["x"].zero_()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        g.replay()
        e1.record()
        noise = torch.randn(4096, device="cuda").square().sum()  # eager work between replays
        torch.cuda.synchronize()
        assert torch.isfinite(noise)
        times.append(e0.elapsed_time(e1))
        assert torch.equal(out["x"], x_e) and torch.equal(out["k"], k_e), f"replay {i} differs from the eager call"
    mk.check()
    _report("whole call graph replays (A)", replays=3, ms=times)


def test_frames_with_ring_append_as_two_graphs_match_eager():
    """Four calls (frames) of modulations + source caches + steps 1..N + register append, replayed as two
    captured graphs, one per buffer parity of the ring (G0 reads set 0 and appends into set 1, G1 the
    reverse): every frame's result equals the eager sequence's, bit for bit, and kv_start evolves on the
    device (from an empty memory: kv_start = PM, then PM - R, ... 0)."""
    from mkx.modulations import ModulationProjection
    from mkx.ring import RegisterRing
    case = make_case(replace(SY.WORKLOADS["A"], kv_start=SY.WORKLOADS["A"].PM))
    cfg, model, past, W = case["cfg"], case["model"], case["past"], case["W"]
    mk = ExpertMegakernel(model)
    prep = SourcePrepare(model)
    proj = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda())
    sc = case["inp"]["state_cond"].cuda()
    ctx = case["inp"]["ctx"].cuda()
    ca_len = torch.tensor([cfg.S], dtype=torch.int32, device="cuda")
    dt = torch.full((1,), -1.0 / cfg.num_steps, device="cuda")
    mem0 = [(k.clone(), v.clone()) for k, v in past.register_step["mem_kv"]]
    ks0 = past.register_step["kv_start"].clone()
    R, T = cfg.R_reg, cfg.T_act
    out = {}

    def call():
        mods = proj(model.modulation_input(cfg.num_steps, sc))[0]
        past.cross_attn_kv = [(k[0], v[0]) for k, v in prep(ctx, ca_len)]
        out["x"], out["k"], out["v"] = mk.run_all(case["noise"], mods, dt, past, cfg.action_dim)

    ring_e = RegisterRing(mem0, ks0, R, kept_delta=-R, new_delta=-(T + R))
    ring_e.update_past(past)
    xs, kss = [], []
    for _ in range(4):
        call()
        xs.append(out["x"].clone())
        ring_e.append_frame(out["k"], out["v"])
        ring_e.update_past(past)
        kss.append(int(ring_e.kv_start[0]))
    mk.check()
    torch.cuda.synchronize()
    assert not torch.equal(xs[0], xs[1])  # the memory changes between frames

    ring_g = RegisterRing(mem0, ks0, R, kept_delta=-R, new_delta=-(T + R))
    ring_g.update_past(past)
    call()  # warm-up (no append: the ring's state is untouched)
    torch.cuda.synchronize()
    graphs, x_of = [], []
    for _ in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call()
            ring_g.append_frame(out["k"], out["v"])
        ring_g.update_past(past)  # the next graph reads the other buffer set
        graphs.append(g)
        x_of.append(out["x"])
    torch.cuda.synchronize()
    for f in range(4):
        graphs[f % 2].replay()
        noise = torch.randn(4096, device="cuda").square().sum()  # eager work between replays
        torch.cuda.synchronize()
        assert torch.isfinite(noise)
        assert torch.equal(x_of[f % 2], xs[f]), f"frame {f} differs from the eager sequence"
        assert int(ring_g._ks[(f + 1) % 2][0]) == kss[f]
    mk.check()
    assert kss == [max(cfg.PM - (f + 1) * R, 0) for f in range(4)]
    _report("frames as two graphs (A)", frames=4, kv_start=kss)


def _source_run(wk, wv, k_norm, ctx, lens, cos, sin, kca, vca, stride):
    """mkx_source_create and mkx_source_run on caller-made buffers: wk, wv [L, NH * 64, C], kca / vca per-layer addresses,
    `stride` elements between samples."""
    L, NH, (B, SP, C) = wk.shape[0], wk.shape[1] // 64, ctx.shape
    lib, stream = _lib.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    h = ctypes.c_void_p()
    dims = _lib.MkxSourceDims(L=L, NH=NH, HD=64, C=C, max_rows=B * SP, eps=1e-6)
    _lib.check(lib.mkx_source_create(ctypes.byref(dims), ctypes.c_void_p(wk.data_ptr()), ctypes.c_void_p(wv.data_ptr()),
                                     ctypes.c_void_p(k_norm.data_ptr()), stream, ctypes.byref(h)), "mkx_source_create")
    a = _lib.MkxSourceArgs(B=B, SP=SP, ctx=ctx.data_ptr(), ca_len=lens.data_ptr(), cos=cos.data_ptr(), sin=sin.data_ptr())
    for l in range(L):
        a.kca[l], a.vca[l] = kca[l], vca[l]
    a.src_stride_b = stride
    _lib.check(lib.mkx_source_run(h, ctypes.byref(a), stream), "mkx_source_run")
    torch.cuda.synchronize()
    lib.mkx_source_destroy(h)


def test_prepare_context_of_four_gigabytes_of_weights_per_head():
    """A context so wide that the byte offsets of a head's weights and of a row group's context pass 2^32. Operands are -1, 0
    and 1, so every partial sum is a whole number below 2^24 and the projections are exact: V is the rounded sum itself."""
    C, SP = (1 << 25) + 96, 20
    g = torch.Generator(device="cuda").manual_seed(3)
    trits = lambda *s: torch.randint(-1, 2, s, generator=g, device="cuda", dtype=torch.int8).bfloat16()  # noqa: E731
    wk, wv, ctx = trits(1, 64, C), trits(1, 64, C), trits(1, SP, C)
    out = torch.full((2, SP, 64), float("nan"), dtype=torch.bfloat16, device="cuda")
    cos, sin = torch.ones(SP, 64, device="cuda"), torch.zeros(SP, 64, device="cuda")
    _source_run(wk, wv, torch.zeros(1, 64, dtype=torch.bfloat16, device="cuda"), ctx,
                torch.tensor([SP], dtype=torch.int32, device="cuda"), cos, sin, [out[0].data_ptr()], [out[1].data_ptr()], SP * 64)
    k, v = torch.zeros(2, SP, 64, dtype=torch.float64, device="cuda")
    for c in range(0, C, 1 << 20):
        x = ctx[0, :, c:c + (1 << 20)].double()
        k += x @ wk[0, :, c:c + (1 << 20)].double().T
        v += x @ wv[0, :, c:c + (1 << 20)].double().T
    assert torch.equal(out[1], v.bfloat16())
    k = k.bfloat16().double()
    k = k * torch.rsqrt((k * k).mean(-1, keepdim=True) + 1e-6)
    # one rounding to bf16 (2^-9) of a value known to a few fp32 roundings
    assert bool(((out[0].double() - k).abs() <= 2.0 ** -8 * k.abs()).all())


@pytest.mark.parametrize("NH, B, SP, C, lens", [
    (3, 3, 37, 160, [37, 0, 20]),                  # odd head count: the last head pair is one head wide
    (1, 5, 31, 96, [0, 31, 0, 17, 0]),             # empty samples first, between and last
    (4, 2, 100, 64, [0, 0]),                       # no valid row at all
    (2, 1, 600, 96, [333]),                        # fewer valid rows than row groups launched
    (3, 64, 5, 64, [(7 * b) % 6 for b in range(64)]),
    (3, 66, 5, 64, [(7 * b) % 6 for b in range(66)]),  # more samples than are numbered densely
    (2, 33, 64, 64, [64 - 2 * b for b in range(33)]),
    (2, 2, 33, 64, [-2, 40]),                      # lengths outside [0, SP]
])
def test_prepare_writes_every_row_and_nothing_else(NH, B, SP, C, lens):
    """Buffers of NaNs with a sample stride past SP * NH * 64 and guards on both sides: rows past a sample's length become
    exactly 0, the others the result, and the gaps and guards stay as they were. One bf16 rounding may move by a unit, and
    the rotation mixes the two halves of a head (the module's tolerances)."""
    L, NAN, G = 2, 0x7FC1, 512
    row = NH * 64
    stride = SP * row + 68
    g = torch.Generator().manual_seed(B)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    wk, wv, kn = (rnd(L, row, C) * 0.1).bfloat16(), (rnd(L, row, C) * 0.1).bfloat16(), (rnd(L, 64) * 0.1).bfloat16()
    ctx = rnd(B, SP, C).bfloat16()
    cos, sin = rope_table(SP, device="cpu")
    buf = torch.full((2, L, G + B * stride + G), NAN, dtype=torch.int16, device="cuda")
    at = lambda i, l: buf[i, l].data_ptr() + 2 * G  # noqa: E731
    _source_run(wk.cuda(), wv.cuda(), kn.cuda(), ctx.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda"), cos.cuda(),
                sin.cuda(), [at(0, l) for l in range(L)], [at(1, l) for l in range(L)], stride)
    buf = buf.cpu()
    body = buf[:, :, G:G + B * stride].view(2, L, B, stride)
    assert bool((buf[:, :, :G] == NAN).all() and (buf[:, :, G + B * stride:] == NAN).all())
    assert bool((body[..., SP * row:] == NAN).all())
    bits = body[..., :SP * row].reshape(2, L, B, SP, NH, 64)
    dead = torch.arange(SP)[None] >= torch.tensor(lens)[:, None]
    assert bool((bits[:, :, dead] == 0).all())
    gk, gv = bits.contiguous().view(torch.bfloat16).double()
    x, live = ctx.double(), ~dead
    for l in range(L):
        v = (x @ wv[l].double().T).bfloat16().double().view(B, SP, NH, 64)
        k = (x @ wk[l].double().T).bfloat16().double().view(B, SP, NH, 64)
        n = (k * torch.rsqrt((k * k).mean(-1, keepdim=True) + 1e-6) * (1 + kn[l].double())).bfloat16().double()
        k = n * cos.double()[:, None] + torch.cat([-n[..., 32:], n[..., :32]], -1) * sin.double()[:, None]
        pair = torch.sqrt(n[..., :32] ** 2 + n[..., 32:] ** 2).repeat(1, 1, 1, 2)
        assert bool(((gv[l] - v).abs() <= 2.0 ** -7 * v.abs() + 2.0 ** -12)[live].all())
        assert bool(((gk[l] - k).abs() <= 2.0 ** -6 * pair + 1e-6)[live].all())
