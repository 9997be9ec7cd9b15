"""GPU: ``mkx_modulations`` (through the C ABI, via mkx.modulations.ModulationProjection) against the CPU
oracle's ``step_modulations`` on the same input c, and the expert run on the kernel's modulation rows.
Tolerance: fp32 products from split-bf16 operands and a hardware exp in SiLU, |delta| <= 1e-4 max|mods|."""
import ctypes
import json
from dataclasses import replace

import pytest
import torch

from _cases import TINY, diff, make_case, oracle_dims, oracle_steps
from mkx import ExpertMegakernel, _lib, synthetic as SY
from mkx.modulations import ModulationProjection, StepModulations
from oracle import expert_ref as ER

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


def _report(name, **kv):
    print(json.dumps({"case": name, **kv}), flush=True)


def _check(name, cfg, n_steps=10):
    W = SY.make_weights(cfg, 0)
    d = oracle_dims(cfg)
    sc = SY.make_inputs(cfg)["state_cond"]
    c = ER.modulation_input(n_steps, sc, W, d)  # [B, N, H]
    ref, _ = ER.step_modulations(n_steps, sc, W, d)
    proj = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda())
    out = proj(c.cuda())
    out_rm = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda(), fragment_order=False)(c.cuda())
    torch.cuda.synchronize()
    assert torch.equal(out, out_rm)  # both weight layouts give the same bits
    dd = (out.cpu() - ref).abs()
    _report(name, max=float(dd.max()), mean=float(dd.mean()), max_abs_ref=float(ref.abs().max()))
    assert out.shape == ref.shape
    assert float(dd.max()) <= 1e-4 * float(ref.abs().max())


def test_modulations_tiny():
    _check("modulations tiny (H 256)", TINY, 4)


def test_modulations_config_A():
    _check("modulations A (L10 H768, 10 steps)", SY.WORKLOADS["A"])


def test_modulations_batch_and_wide():
    _check("modulations B8 (80 rows)", SY.WORKLOADS["B"])
    _check("modulations D shape (L16 H1024)", replace(SY.WORKLOADS["D"], weight_dtype="bf16"))


def test_expert_on_kernel_modulations():
    case = make_case(SY.WORKLOADS["A"])
    cfg, model = case["cfg"], case["model"]
    W = case["W"]
    c = ER.modulation_input(cfg.num_steps, case["inp"]["state_cond"], W, oracle_dims(cfg))
    mods_k = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda())(c.cuda())[0]  # [N, MODW], B = 1
    mk = ExpertMegakernel(model)
    x_t, _, _ = mk.run_all(case["noise"], case["mods"], case["dt"], case["past"], cfg.action_dim)
    x_k, _, _ = mk.run_all(case["noise"], mods_k, case["dt"], case["past"], cfg.action_dim)
    mk.check()
    torch.cuda.synchronize()
    case_k = dict(case, mods=mods_k)
    r32 = oracle_steps(case_k, case["noise"], 0, cfg.num_steps, "fp32", first=True)
    m, a = diff(x_k, r32, cfg.action_dim)
    mt, _ = diff(x_k, x_t, cfg.action_dim)
    _report("expert on kernel modulations (A)", vs_fp32_max=m, vs_fp32_mean=a, vs_torch_mods_max=mt)
    assert m <= 1e-3 and a <= 2e-4 and mt <= 1e-3


def test_modulations_timing_config_A():
    """Kernel vs the PyTorch projection (fp32 weights) on config A's 10 rows; reported, not asserted."""
    cfg = SY.WORKLOADS["A"]
    W = SY.make_weights(cfg, 0)
    c = ER.modulation_input(cfg.num_steps, SY.make_inputs(cfg)["state_cond"], W, oracle_dims(cfg)).cuda()
    proj = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda())
    wf, bf = W["mod_w"].float().cuda(), W["mod_b"].float().cuda()

    def t(fn, n=50):
        for _ in range(3):
            fn()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for _ in range(n):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) * 1e3 / n

    proj_rm = ModulationProjection(W["mod_w"].cuda(), W["mod_b"].float().cuda(), fragment_order=False)
    _report("modulations timing A", kernel_us=t(lambda: proj(c)), kernel_row_major_us=t(lambda: proj_rm(c)),
            torch_fp32_us=t(lambda: torch.nn.functional.silu(c) @ wf.T + bf),
            weight_bytes=int(proj.w.numel() * 2))


def _step_mods(W):
    return StepModulations(W["t1_w"].cuda(), W["t1_b"].cuda(), W["t2_w"].cuda(), W["t2_b"].cuda(), W["mod_w"].cuda(),
                           W["mod_b"].cuda())


def _check_input(name, cfg, n_steps):
    """mkx_modulation_input (timestep embedding and the small MLP) against the oracle's modulation_input,
    then the whole _step_modulations (input kernel + projection) against the oracle's step_modulations:
    fp32 products from split-bf16 operands and a hardware exp in SiLU, |delta| <= 1e-4 of the largest value."""
    W = SY.make_weights(cfg, 0)
    d = oracle_dims(cfg)
    sc = SY.make_inputs(cfg)["state_cond"]
    sm = _step_mods(W)
    c = sm.input(n_steps, sc.cuda())
    ref_c = ER.modulation_input(n_steps, sc, W, d)
    mods, dt = sm(n_steps, sc.cuda())
    ref, ref_dt = ER.step_modulations(n_steps, sc, W, d)
    torch.cuda.synchronize()
    ref = ref[0] if cfg.B == 1 else ref
    dc, dm = (c.cpu() - ref_c).abs(), (mods.cpu() - ref).abs()
    _report(name, c_max=float(dc.max()), c_max_abs_ref=float(ref_c.abs().max()), mods_max=float(dm.max()),
            mods_max_abs_ref=float(ref.abs().max()))
    assert c.shape == ref_c.shape and mods.shape == ref.shape
    assert float(dc.max()) <= 1e-4 * float(ref_c.abs().max())
    assert float(dm.max()) <= 1e-4 * float(ref.abs().max())
    assert float(dt.item()) == pytest.approx(ref_dt)


def test_modulation_input_tiny():
    _check_input("modulation input tiny (H 256, tdim 32)", TINY, TINY.num_steps)


def test_modulation_input_config_A():
    _check_input("modulation input A (10 steps)", SY.WORKLOADS["A"], 10)


def test_modulation_input_batch_of_8():
    _check_input("modulation input B (8 samples)", SY.WORKLOADS["B"], 10)


def test_modulation_input_one_step_and_two_row_tiles():
    _check_input("modulation input A, 1 step", SY.WORKLOADS["A"], 1)
    _check_input("modulation input A, 20 steps (two row tiles)", SY.WORKLOADS["A"], 20)


def test_modulation_input_wide_expert():
    _check_input("modulation input D shape (H 1024)", replace(SY.WORKLOADS["D"], L=2), 10)


def test_step_modulations_drive_the_expert_like_the_pytorch_ones():
    """The expert run (Euler steps 1..N in one launch) on the kernels' modulation rows against the run on the
    synthetic model's PyTorch rows: the same up to the modulations' rounding."""
    cfg = SY.WORKLOADS["A"]
    case = make_case(cfg)
    model, past, noise = case["model"], case["past"], case["noise"]
    mk = ExpertMegakernel(model)
    sc = case["inp"]["state_cond"].cuda()
    mods_k, dt_k = _step_mods(case["W"])(cfg.num_steps, sc)
    mods_t, dt_t = model._step_modulations(cfg.num_steps, sc)
    x_k, _, _ = mk.run_all(noise, mods_k, dt_k, past, cfg.action_dim)
    x_t, _, _ = mk.run_all(noise, mods_t, dt_t, past, cfg.action_dim)
    mk.check()
    torch.cuda.synchronize()
    m, a = diff(x_k, x_t, cfg.action_dim)
    _report("expert on kernel step modulations vs PyTorch step modulations (A)", max=m, mean=a)
    assert m <= 1e-3 and a <= 2e-4


def _rand(*shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g) * std


@pytest.mark.parametrize("fragment_order", [True, False])
@pytest.mark.parametrize("R, K, N", [(1, 256, 16), (16, 768, 48), (17, 512, 4112), (33, 1024, 16 * 300), (48, 768, 16 * 257),
                                     (49, 256, 16 * 513), (65, 768, 16 * 1030), (80, 1024, 16 * 700), (81, 512, 32),
                                     (129, 768, 16 * 259), (161, 1024, 16)])
def test_modulations_row_and_column_edges(R, K, N, fragment_order):
    """Row tiles of every count a workgroup holds and more than one row group; fewer column tiles than workgroups,
    and ranges that leave remainders of the weights' pipeline. Against 64 bits: silu(c) is held in three
    bf16 parts (well within the 2^-18 of two), a result is a sum of at most 3 K / 8 + 16 fp32 additions per wave and
    over the waves, each rounded to 2^-24 of at most S = sum |silu(c) w| + |b|; the hardware exp and reciprocal add 2^-20."""
    c, w, b = _rand(R, K + 12, seed=R)[:, :K], _rand(N, K, seed=K, std=0.02).bfloat16(), _rand(N, seed=N, std=0.02)
    proj = ModulationProjection(w.cuda(), b.cuda(), fragment_order=fragment_order)
    out = proj(c.cuda()).cpu().double()
    a = torch.nn.functional.silu(c.double())
    ref = a @ w.double().T + b.double()
    S = a.abs() @ w.double().abs().T + b.double().abs()
    bound = (2.0 ** -18 + 2.0 ** -20 + (3 * K / 8 + 16) * 2.0 ** -24) * S
    assert bool(((out - ref).abs() <= bound).all()), float(((out - ref).abs() / S).max())


@pytest.mark.parametrize("K", [256, 512, 768, 1024])
def test_modulations_rows_do_not_depend_on_their_number(K):
    """A row's result is the same bits alone and among any number of rows (row tiles per workgroup and row groups differ)."""
    w, b = _rand(16 * 259, K, seed=K, std=0.02).bfloat16(), _rand(16 * 259, seed=9, std=0.02)
    c = _rand(161, K, seed=10).cuda()
    proj = ModulationProjection(w.cuda(), b.cuda())
    whole = proj(c)
    for R in (1, 10, 17, 48, 49, 64, 65, 80, 81, 96, 97, 113, 128, 160):
        assert torch.equal(proj(c[:R]), whole[:R]), R


def _input_single_launch(step, N, sc):
    """mkx_modulation_input, the entry without a workspace, on the weights of a StepModulations."""
    sc = sc.cuda()
    out = torch.empty(sc.shape[0], N, step.H, device="cuda")
    a = _lib.MkxModinArgs(N=N, B=sc.shape[0], H=step.H, tdim=step.tdim, t1_w=step.t1_w.data_ptr(), t1_b=step.t1_b.data_ptr(),
                          t2_w=step.t2_w.data_ptr(), t2_b=step.t2_b.data_ptr(), state_cond=sc.data_ptr(), sc_stride=step.H,
                          out=out.data_ptr(), out_stride_b=N * step.H, out_stride_k=step.H)
    _lib.check(_lib.lib().mkx_modulation_input(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "mkx_modulation_input")
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("N, B, H, tdim", [(1, 1, 256, 32), (10, 1, 768, 256), (15, 5, 512, 64), (16, 2, 768, 160), (17, 3, 1024, 512),
                                           (33, 6, 1024, 96)])
def test_modulation_input_step_and_width_edges(N, B, H, tdim, workspace):
    """Steps below, at and past a row tile of 16, every width, odd k-block counts of the embedding and more samples than
    waves share a column tile. Against 64 bits, with the error carried through: embedding rounded to fp32 (2^-24), sums of
    n fp32 additions (n 2^-24 of the sum of magnitudes), silu (slope at most 1.1; hardware exp 2^-20)."""
    bf = torch.bfloat16
    t1w, t2w = _rand(H, tdim, seed=1, std=0.05).to(bf), _rand(H, H, seed=2, std=0.05).to(bf)
    t1b, t2b, sc = _rand(H, seed=3, std=0.1), _rand(H, seed=4, std=0.1), _rand(B, H, seed=5)
    step = StepModulations(t1w.cuda(), t1b.cuda(), t2w.cuda(), t2b.cuda(), _rand(16, H, seed=6).to(bf).cuda(), _rand(16, seed=7).cuda())
    out = (step.input(N, sc.cuda()) if workspace else _input_single_launch(step, N, sc)).cpu().double()
    d = torch.float64
    half = tdim // 2
    arg = 1000.0 * (1.0 - torch.arange(N, dtype=d) / N)[:, None] * 10000.0 ** (-torch.arange(half, dtype=d) / half)
    temb = torch.cat([torch.cos(arg), torch.sin(arg)], -1)
    pre = temb @ t1w.to(d).T + t1b.to(d)
    h1 = torch.nn.functional.silu(pre)
    ref = (h1 @ t2w.to(d).T + t2b.to(d))[None] + sc.to(d)[:, None]
    e_pre = (3 * tdim + 8) * 2.0 ** -24 * (temb.abs() @ t1w.to(d).abs().T + t1b.to(d).abs())
    e_h1 = 1.1 * e_pre + 2.0 ** -20 * h1.abs()
    bound = e_h1 @ t2w.to(d).abs().T + (3 * H / 4 + 16) * 2.0 ** -24 * (h1.abs() @ t2w.to(d).abs().T + t2b.to(d).abs())
    bound = bound[None] + 2.0 ** -22 * (1.0 + sc.to(d).abs()[:, None])
    assert bool(((out - ref).abs() <= bound).all()), float((out - ref).abs().max())


@pytest.mark.parametrize("R, K, N", [(3, 256, 48), (20, 768, 16 * 300), (70, 512, 64), (70, 1024, 64), (100, 768, 32)])
def test_modulations_padded_strides(R, K, N):
    """Rows of c and of the result further apart than they are long: the same bits as with dense rows, nothing read from
    the gaps (NaNs) and nothing written to them."""
    w, b = _rand(N, K, seed=K, std=0.02).bfloat16().cuda(), _rand(N, seed=N, std=0.02).cuda()
    dense = _rand(R, K, seed=R).cuda()
    want = ModulationProjection(w, b, fragment_order=False)(dense)
    cs, os_ = K + 20, N + 12
    c, out = torch.full((R, cs), float("nan"), device="cuda"), torch.full((R + 1, os_), float("nan"), device="cuda")
    c[:, :K] = dense
    a = _lib.MkxModprojArgs(R=R, K=K, N=N, c=c.data_ptr(), c_stride=cs, w=w.data_ptr(), bias=b.data_ptr(), out=out.data_ptr(),
                            out_stride=os_, w_fragment_order=0)
    _lib.check(_lib.lib().mkx_modulations(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
               "mkx_modulations")
    torch.cuda.synchronize()
    assert torch.equal(out[:R, :N], want)
    assert bool(torch.isnan(out[:, N:]).all() and torch.isnan(out[R]).all())


@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("N, B, H, tdim", [(1, 1, 256, 32), (10, 3, 768, 256), (17, 2, 512, 96), (16, 5, 1024, 512)])
def test_modulation_input_padded_strides(N, B, H, tdim, workspace):
    """state_cond rows, steps and samples further apart than dense: the same bits, gaps neither read nor written, and no
    float past the workspace's N * H."""
    bf = torch.bfloat16
    t1w, t2w = _rand(H, tdim, seed=1, std=0.05).to(bf).cuda(), _rand(H, H, seed=2, std=0.05).to(bf).cuda()
    t1b, t2b, sc = _rand(H, seed=3, std=0.1).cuda(), _rand(H, seed=4, std=0.1).cuda(), _rand(B, H, seed=5).cuda()
    lib, stream = _lib.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(s, out, sc_stride, sb, sk):
        a = _lib.MkxModinArgs(N=N, B=B, H=H, tdim=tdim, t1_w=t1w.data_ptr(), t1_b=t1b.data_ptr(), t2_w=t2w.data_ptr(),
                              t2_b=t2b.data_ptr(), state_cond=s.data_ptr(), sc_stride=sc_stride, out=out.data_ptr(),
                              out_stride_b=sb, out_stride_k=sk)
        if workspace:
            ws = torch.full((N * H + 64,), float("nan"), device="cuda")
            _lib.check(lib.mkx_modulation_input_ws(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), stream), "mkx_modulation_input_ws")
            torch.cuda.synchronize()
            assert bool(torch.isfinite(ws[:N * H]).all() and torch.isnan(ws[N * H:]).all())
        else:
            _lib.check(lib.mkx_modulation_input(ctypes.byref(a), stream), "mkx_modulation_input")
            torch.cuda.synchronize()
        return out

    want = run(sc, torch.empty(B, N, H, device="cuda"), H, N * H, H)
    cs, sk, pad = H + 8, H + 20, 36
    wide = torch.full((B, cs), float("nan"), device="cuda")
    wide[:, :H] = sc
    got = run(wide, torch.full((B + 1, N * sk + pad), float("nan"), device="cuda"), cs, N * sk + pad, sk)
    rows = got[:B, :N * sk].view(B, N, sk)
    assert torch.equal(rows[..., :H], want)
    assert bool(torch.isnan(rows[..., H:]).all() and torch.isnan(got[:, N * sk:]).all() and torch.isnan(got[B]).all())
