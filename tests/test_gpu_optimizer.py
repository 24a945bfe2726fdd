"""GPU parity of FusedAdamW on the BASELINE configs, against the oracle and torch.

  config 1: 6 FP32 tensors, 10 steps, wd .1 on 2-D only (param groups);
  config 2: the 5B SwiGLU stage window, FP16 grads x 2^16, FP16 export;
  config 3: the tied 65536 x 3072 embedding, sparse Zipf rows, BF16 grads/export, wd 0;
  config 4: config 2 for 16 steps with inf/NaN injected at steps 3, 7, 12.
Bit-exact against the oracle everywhere; against torch.optim.AdamW the moments
are bit-exact and masters agree to max|dw|/max|w| <= 1e-6 (torch's CPU sqrt is
not correctly rounded; see tests/test_oracle_adamw.py).
"""
import copy
import json

import numpy as np
import pytest
import torch

import bench
from morph_amd import DynamicLossScale, FusedAdamW
from tests.golden.make_golden import CONFIG1, config1_inputs, sha
from tests.helpers import assert_same_bits, export_bits, to_oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def oracle_adamw_threads(grad, w, m, v, hp, out_dtype, grad_dtype, parts=16):
    """The oracle's AdamW over `parts` slices on host threads.  Every element's arithmetic
    is its own, so the result is a single call's bit for bit; ctypes releases the GIL
    during the call, which brings a full-size config-3 step to about a second."""
    from concurrent.futures import ThreadPoolExecutor
    from oracle import reference as R
    n = w.size
    if n < (1 << 22):
        return R.adamw(grad, w, m, v, hp, out_dtype=out_dtype, grad_dtype=grad_dtype)
    cuts = [n * k // parts for k in range(parts + 1)]

    def one(k):
        lo, hi = cuts[k], cuts[k + 1]
        return R.adamw(grad[lo:hi], w[lo:hi], m[lo:hi], v[lo:hi], hp, out_dtype=out_dtype,
                       grad_dtype=grad_dtype)

    with ThreadPoolExecutor(parts) as pool:
        outs = list(pool.map(one, range(parts)))
    return None if outs[0] is None else np.concatenate(outs)


class OracleWindow:
    """The oracle's view of a window: one (w, m, v, clock) per tensor."""

    def __init__(self, masters):
        self.w = [to_oracle(t).copy() for t in masters]
        self.m = [np.zeros_like(w) for w in self.w]
        self.v = [np.zeros_like(w) for w in self.w]
        self.t = [0] * len(self.w)

    def step(self, grads, hps_for, out_dtype):
        from oracle import reference as R
        outs = []
        for i, g in enumerate(grads):
            self.t[i] += 1
            outs.append(oracle_adamw_threads(
                to_oracle(g), self.w[i], self.m[i], self.v[i], hps_for(i, self.t[i]), out_dtype,
                {torch.float16: R.DTYPE_F16, torch.bfloat16: R.DTYPE_BF16,
                 torch.float32: R.DTYPE_F32}[g.dtype]))
        return outs

    def check(self, opt, what):
        for i, p in enumerate(p for g in opt.param_groups for p in g["params"]):
            st = opt.state[p]
            assert_same_bits(p.detach().cpu().numpy().ravel(), self.w[i], f"{what} master[{i}]")
            assert_same_bits(st["exp_avg"].cpu().numpy().ravel(), self.m[i], f"{what} m[{i}]")
            assert_same_bits(st["exp_avg_sq"].cpu().numpy().ravel(), self.v[i], f"{what} v[{i}]")
            assert st["step"] == self.t[i]


def test_config1_bitexact_vs_oracle_and_torch_golden(golden_dir):
    from oracle import reference as R
    ref = json.loads((golden_dir / "config1.json").read_text())
    masters, grads = config1_inputs()
    dev = [m.to(DEV) for m in masters]
    groups = [dict(params=[p for p in dev if p.ndim == 2], weight_decay=CONFIG1["wd_2d"]),
              dict(params=[p for p in dev if p.ndim == 1], weight_decay=0.0)]
    opt = FusedAdamW(groups, lr=CONFIG1["lr"], betas=CONFIG1["betas"], eps=CONFIG1["eps"],
                     sync=True)
    order = [p for g in opt.param_groups for p in g["params"]]
    index = [next(i for i, q in enumerate(dev) if q is p) for p in order]
    ora = OracleWindow([masters[i] for i in index])
    for t in range(1, CONFIG1["steps"] + 1):
        gs = grads(t)
        assert opt.step([gs[i].to(DEV) for i in index]) is True
        ora.step([gs[i] for i in index],
                 lambda i, step: R.torch_adamw_hp(CONFIG1["lr"], *CONFIG1["betas"], CONFIG1["eps"],
                                                  CONFIG1["wd_2d"] if order[i].ndim == 2 else 0.,
                                                  step), R.DTYPE_NONE)
    ora.check(opt, "config1")
    for k, i in enumerate(index):  # torch.optim.AdamW golden: moments by SHA, masters sampled
        tref = ref["tensors"][i]
        st = opt.state[order[k]]
        assert sha(st["exp_avg"].cpu().numpy().ravel()) == tref["sha_m"]
        assert sha(st["exp_avg_sq"].cpu().numpy().ravel()) == tref["sha_v"]
        w = order[k].detach().cpu().numpy().ravel()
        idx = np.array(tref["sample_index"])
        assert np.abs(w[idx] - np.array(tref["sample_w"], np.float32)).max() <= 1e-6 * np.abs(w).max()


def test_config1_vs_live_torch_adamw_on_gpu_box():
    """torch.optim.AdamW(foreach=False) on this host's CPU, element by element."""
    masters, grads = config1_inputs()
    ref = [torch.nn.Parameter(m.clone()) for m in masters]
    tgroups = [dict(params=[p for p in ref if p.ndim == 2], weight_decay=.1),
               dict(params=[p for p in ref if p.ndim == 1], weight_decay=0.)]
    topt = torch.optim.AdamW(tgroups, lr=3e-4, betas=(.9, .95), eps=1e-8, foreach=False)
    dev = [m.to(DEV) for m in masters]
    groups = [dict(params=[p for p in dev if p.ndim == 2], weight_decay=.1),
              dict(params=[p for p in dev if p.ndim == 1], weight_decay=0.)]
    opt = FusedAdamW(groups, lr=3e-4, betas=(.9, .95), eps=1e-8)  # asynchronous steps
    for t in range(1, 11):
        gs = grads(t)
        for p, g in zip(ref, gs):
            p.grad = g.clone()
        topt.step()
        by_id = {id(p): g for p, g in zip(dev, gs)}
        opt.step([by_id[id(p)].to(DEV) for grp in opt.param_groups for p in grp["params"]])
    opt.resolve()
    for p, q in zip(ref, dev):
        st, qs = topt.state[p], opt.state[q]
        assert torch.equal(st["exp_avg"], qs["exp_avg"].cpu())
        assert torch.equal(st["exp_avg_sq"], qs["exp_avg_sq"].cpu())
        dw = (q.detach().cpu() - p.detach()).abs().max() / p.detach().abs().max()
        assert dw <= 1e-6
        assert int(qs["step"]) == int(st["step"]) == 10


def _config2_run(shapes, steps, seed, check_at=()):
    from oracle import reference as R
    masters = [m.cpu() for m in bench.config2_window("cpu", seed)] if shapes is None else [
        torch.randn(s, generator=torch.Generator().manual_seed(seed + i)) * .02
        for i, s in enumerate(shapes)]
    shapes = [tuple(m.shape) for m in masters]
    scaler = DynamicLossScale(65536., 2000)
    opt = FusedAdamW([m.to(DEV) for m in masters], lr=3e-4, betas=(.9, .95), eps=1e-8,
                     weight_decay=.1, loss_scale=scaler, export_dtype=torch.float16, sync=True)
    ora = OracleWindow(masters)
    outs = None
    for t in range(1, steps + 1):
        grads = bench.config2_grads("cpu", 1000 + t, shapes)
        assert opt.step([g.to(DEV) for g in grads]) is True
        outs = ora.step(grads, lambda i, step: R.torch_adamw_hp(3e-4, .9, .95, 1e-8, .1, step,
                                                                scale=65536.), R.DTYPE_F16)
        if t in check_at or t == steps:
            ora.check(opt, f"config2 step {t}")
            for i, o in enumerate(outs):
                assert_same_bits(export_bits(opt.exports[i]), o.view(np.uint16),
                                 f"step {t} export[{i}]")
            print(f"config 2 step {t}: masters, moments, export bit-exact", flush=True)
    assert scaler.scale == 65536. and scaler.good_steps == steps


def test_config2_window_reduced_20_steps():
    _config2_run([(768, 384), (768, 384), (384, 768)], steps=20, seed=3)


def test_config2_window_full_size_20_steps():
    """BASELINE config 2 as stated: N = 56,623,104 at the real shapes, 20 steps, bit-exact
    vs the oracle at step 10 and at the end (masters, moments, clocks, FP16 export)."""
    _config2_run(None, steps=20, seed=0, check_at=(10,))


def test_config3_tied_embedding_full_size_20_steps():
    """BASELINE config 3 as stated: [65536, 3072] BF16 sparse-row grads (a fresh Zipf draw
    per step), wd 0, BF16 export, 20 steps; every row decays/updates.  Bit-exact vs the
    oracle at step 10 and at the end."""
    from oracle import reference as R
    w0 = torch.randn(65536, 3072, generator=torch.Generator().manual_seed(4)) * .02
    opt = FusedAdamW([w0.to(DEV)], lr=3e-4, betas=(.9, .95), eps=1e-8, weight_decay=0.0,
                     export_dtype=torch.bfloat16, sync=True)
    ora = OracleWindow([w0])
    for t in range(1, 21):
        g, active = bench.config3_embedding_grad(7000 + t)
        assert 100 < active.numel() < 4096
        assert opt.step([g.to(DEV)]) is True
        outs = ora.step([g], lambda i, step: R.torch_adamw_hp(3e-4, .9, .95, 1e-8, 0.0, step),
                        R.DTYPE_BF16)
        del g
        if t in (10, 20):
            ora.check(opt, f"config3 step {t}")
            assert_same_bits(export_bits(opt.exports[0]), outs[0], f"step {t} export")
            print(f"config 3 step {t}: masters, moments, export bit-exact", flush=True)
    # property: a row that never had a gradient keeps m = v = 0 and w = w0 exactly
    p = opt.param_groups[0]["params"][0]
    st = opt.state[p]
    zero_rows = (st["exp_avg_sq"].abs().sum(1) == 0).nonzero().flatten()[:64].cpu()
    assert zero_rows.numel() > 0
    assert torch.equal(p.detach()[zero_rows.to(DEV)].cpu(), w0[zero_rows])


@pytest.mark.parametrize("shapes", [[(768, 384), (768, 384), (384, 768)], None],
                         ids=["reduced", "full"])
def test_config4_overflow_skip_sequence(golden_dir, shapes):
    """Skip decisions, untouched state on skipped steps and the scale sequence, bit-exact."""
    from oracle import reference as R
    cfg = json.loads((golden_dir / "loss_scale.json").read_text())["config4"]
    if shapes is None:
        masters = bench.config2_window("cpu", 0)
    else:
        masters = [torch.randn(s, generator=torch.Generator().manual_seed(20 + i)) * .02
                   for i, s in enumerate(shapes)]
    shapes = [tuple(m.shape) for m in masters]
    scaler = DynamicLossScale(cfg["initial"], cfg["growth_interval"])
    oscaler = R.LossScale(cfg["initial"], cfg["growth_interval"])
    opt = FusedAdamW([m.to(DEV) for m in masters], lr=3e-4, betas=(.9, .95), eps=1e-8,
                     weight_decay=.1, loss_scale=scaler, export_dtype=torch.float16, sync=True)
    ora = OracleWindow(masters)
    rng = np.random.RandomState(44)
    seen = []
    for t in range(1, cfg["steps"] + 1):
        seen.append(scaler.scale)
        assert scaler.scale == oscaler.scale
        grads = bench.config2_grads("cpu", 2000 + t, shapes, scale=scaler.scale)
        if t in cfg["overflow_steps"]:
            for _ in range(int(rng.randint(1, 9))):
                k = int(rng.randint(len(grads)))
                flat = grads[k].view(-1)
                flat[int(rng.randint(flat.numel()))] = float(rng.choice([np.inf, -np.inf, np.nan]))
        decision = any(R.nonfinite_any(to_oracle(g)) for g in grads)
        before = [p.detach().clone() for p in opt.param_groups[0]["params"]]
        before_exp = [e.clone() for e in opt.exports]
        applied = opt.step([g.to(DEV) for g in grads])
        assert applied is (not decision)
        if decision:
            oscaler.overflow()
            for p, b in zip(opt.param_groups[0]["params"], before):
                assert torch.equal(p, b)
            for e, b in zip(opt.exports, before_exp):
                assert torch.equal(e, b)
        else:
            oscaler.success()
            sc = seen[-1]
            ora.step(grads, lambda i, step: R.torch_adamw_hp(3e-4, .9, .95, 1e-8, .1, step,
                                                             scale=sc), R.DTYPE_F16)
    assert seen == cfg["scale_before_step"]
    assert scaler.state_dict() == oscaler.state_dict()
    assert opt.skipped_steps == len(cfg["overflow_steps"])
    ora.check(opt, "config4")


def test_none_grad_leaves_param_and_clock():
    """sparse_disk.py:1-5: no gradient -> no update, no clock advance."""
    a = torch.randn(1000, generator=torch.Generator().manual_seed(1)).to(DEV)
    b = torch.randn(1000, generator=torch.Generator().manual_seed(2)).to(DEV)
    b0 = b.clone()
    opt = FusedAdamW([a, b], lr=1e-3, sync=True)
    g = torch.randn(1000, device=DEV) * 1e-3
    assert opt.step([g, None])
    assert opt.step([g, None])
    assert opt.state[a]["step"] == 2 and opt.state[b]["step"] == 0
    assert torch.equal(b, b0)
    assert opt.step([None, g])
    assert opt.state[b]["step"] == 1


def test_state_dict_interchanges_with_torch_adamw():
    """A torch.optim.AdamW state dict loads into FusedAdamW and the runs continue identically."""
    gen = torch.Generator().manual_seed(6)
    w = torch.randn(5000, generator=gen) * .02
    grads = [torch.randn(5000, generator=gen) * 1e-3 for _ in range(4)]
    p = torch.nn.Parameter(w.clone())
    topt = torch.optim.AdamW([p], lr=1e-3, betas=(.9, .95), weight_decay=.1, foreach=False)
    for g in grads[:2]:
        p.grad = g.clone()
        topt.step()
    q = p.detach().clone().to(DEV)
    opt = FusedAdamW([q], lr=1e-3, betas=(.9, .95), weight_decay=.1)
    sd = topt.state_dict()
    opt.load_state_dict(sd)
    assert opt.state[q]["step"] == 2
    for g in grads[2:]:
        p.grad = g.clone()
        topt.step()
        opt.step([g.to(DEV)])
    opt.resolve()
    assert opt.state[q]["step"] == 4
    assert torch.equal(opt.state[q]["exp_avg"].cpu(), topt.state[p]["exp_avg"])
    assert torch.equal(opt.state[q]["exp_avg_sq"].cpu(), topt.state[p]["exp_avg_sq"])
    assert (q.cpu() - p.detach()).abs().max() <= 1e-6 * p.detach().abs().max()
    back = opt.state_dict()
    assert float(back["state"][0]["step"]) == 4.0



def test_arena_layout_gives_identical_steps():
    """arena=True moves masters, moments and exports into one allocation: the steps,
    the exports and the state dict are bit-identical to separate allocations, and each
    parameter object keeps its identity with its data in the arena."""
    shapes = [(1024, 1024), (3072,), (768, 384), (2048, 1024), (5,)]
    gen = torch.Generator().manual_seed(70)
    masters = [torch.randn(s, generator=gen) * .02 for s in shapes]
    grads = [[(torch.randn(s, generator=gen) * 1e-4 * 1024).half() for s in shapes]
             for _ in range(3)]
    runs = []
    for arena in (False, True):
        params = [torch.nn.Parameter(m.to(DEV)) for m in masters]
        groups = [{"params": params[:2], "weight_decay": .1}, {"params": params[2:]}]
        opt = FusedAdamW(groups, lr=3e-4, betas=(.9, .95), eps=1e-8, weight_decay=0.0,
                         loss_scale=1024.0, export_dtype=torch.float16, arena=arena)
        for p, m in zip(params, masters):
            assert torch.equal(p.detach().cpu(), m)
        if arena:
            base, end = opt.arena.storage.data_ptr(), opt.arena.storage.data_ptr() + opt.arena.nbytes
            for p in params:
                for t in (p, opt.state[p]["exp_avg"], opt.state[p]["exp_avg_sq"]):
                    assert base <= t.data_ptr() < end
        for gs in grads:
            opt.step([g.to(DEV) for g in gs])
        opt.resolve()
        runs.append((params, opt))
    (pa, a), (pb, b) = runs
    for p, q in zip(pa, pb):
        assert torch.equal(p, q)
        for k in ("exp_avg", "exp_avg_sq"):
            assert torch.equal(a.state[p][k], b.state[q][k])
        assert a.state[p]["step"] == b.state[q]["step"] == 3
    for e, f in zip(a.exports, b.exports):
        assert torch.equal(e, f)
    sa, sb = a.state_dict(), b.state_dict()
    for i in sa["state"]:
        assert torch.equal(sa["state"][i]["exp_avg_sq"], sb["state"][i]["exp_avg_sq"])


def test_new_gradient_buffers_swap_pointers_only():
    """A new gradient buffer every step (autograd with set_to_none) reuses the launch
    table with swapped pointers and gives the same bytes as one reused buffer; a size
    mismatch is rejected before anything is enqueued."""
    shapes = [(300, 70), (4099,)]
    gen = torch.Generator().manual_seed(71)
    masters = [torch.randn(s, generator=gen) * .02 for s in shapes]
    grads = [[torch.randn(s, generator=gen).half() for s in shapes] for _ in range(4)]
    a = FusedAdamW([m.to(DEV) for m in masters], lr=1e-3, loss_scale=8.0)
    b = FusedAdamW([m.to(DEV) for m in masters], lr=1e-3, loss_scale=8.0)
    held = [g.to(DEV) for g in grads[0]]
    tables = set()
    for gs in grads:
        a.step([g.to(DEV) for g in gs])
        tables.add(id(a._cache[0]))
        for h, g in zip(held, gs):
            h.copy_(g.to(DEV))
        b.step(held)
    a.resolve()
    b.resolve()
    assert len(tables) == 1
    for p, q in zip(a.param_groups[0]["params"], b.param_groups[0]["params"]):
        assert torch.equal(p, q)
        assert torch.equal(a.state[p]["exp_avg_sq"], b.state[q]["exp_avg_sq"])
    with pytest.raises(ValueError):
        a._cache[0].rebind_grads([torch.zeros(10, dtype=torch.half, device=DEV), held[1]])


@pytest.mark.parametrize("prev_inf,now_inf,scale,count", [
    (0, 0, 1024.0, 2), (1, 0, 1024.0, 2), (0, 1, 1024.0, 2), (1, 1, 1024.0, 2),
    (1, 0, 1.0, 2), (0, 0, 2.0 ** 15, 0), (1, 0, 512.0, 0)],
    ids=["clean", "prev-overflow", "now-overflow", "both", "fatal", "close-only", "close-only-inf"])
def test_fused_detector_close_equals_separate_launches(prev_inf, now_inf, scale, count):
    """morph_nonfinite_or_close(slot) leaves the state block and the clocks byte-identical
    to morph_step_end(slot ^ 1) followed by the detector into found_inf[slot]."""
    from morph_amd import kernels
    from morph_amd.control import StepControl
    gen = torch.Generator().manual_seed(80)
    grads = [torch.randn(1000 + 37 * k, generator=gen).half() for k in range(count)]
    if now_inf:
        grads[0][17] = float("inf")
    grads = [g.to(DEV) for g in grads]
    blocks = []
    for fused in (False, True):
        ctl = StepControl(DEV, 4, DynamicLossScale(scale, growth_interval=3))
        st = ctl.read()
        st.good_steps = 2  # the next success grows the scale
        st.found_inf[1] = prev_inf
        ctl.state.copy_(torch.frombuffer(bytearray(bytes(st)), dtype=torch.uint8))
        ctl.clocks.copy_(torch.tensor([5, 6, 7, 8]))
        clock_list = torch.tensor([0, 2, 3], dtype=torch.int32, device=DEV)
        if fused:
            kernels.nonfinite_or_close(grads, ctl.state, 0, ctl.clocks, clock_list)
        else:
            kernels.step_end(ctl.state, ctl.clocks, clock_list, slot=1)
            kernels.nonfinite_or(grads, ctl.found_inf_ptr(0))
        torch.cuda.synchronize()
        blocks.append((ctl.state.cpu(), ctl.clocks.cpu(), ctl.read()))
    (sa, ca, a), (sb, cb, b) = blocks
    assert torch.equal(sa, sb) and torch.equal(ca, cb)
    assert b.found_inf[0] == now_inf and b.found_inf[1] == 0
    assert b.last_found_inf == prev_inf
    if prev_inf and scale <= 1.0:
        assert b.fatal == 1 and cb.tolist() == [5, 6, 7, 8]
    elif prev_inf:
        assert b.scale == scale / 2 and b.skipped == 1 and cb.tolist() == [5, 6, 7, 8]
    else:
        assert b.scale == min(2 * scale, 65536.0) and b.applied == 1
        assert cb.tolist() == [6, 6, 8, 9]


def test_steps_on_alternating_streams_equal_one_stream(golden_dir):
    """A pending step close is enqueued on the stream of its own step when the next step
    runs on another stream: 16 config-4 steps alternating between two streams (each
    waiting for the other) end where the step-by-step run ends."""
    cfg = json.loads((golden_dir / "loss_scale.json").read_text())["config4"]
    shapes = [(512, 256), (1000,)]
    masters = [torch.randn(s, generator=torch.Generator().manual_seed(90 + i)) * .02
               for i, s in enumerate(shapes)]
    streams = [torch.cuda.Stream(DEV), torch.cuda.Stream(DEV)]
    runs = []
    for alternate in (False, True):
        scaler = DynamicLossScale(cfg["initial"], cfg["growth_interval"])
        opt = FusedAdamW([m.to(DEV) for m in masters], lr=3e-4, betas=(.9, .95),
                         weight_decay=.1, loss_scale=scaler, export_dtype=torch.float16,
                         sync=not alternate)
        rng = np.random.RandomState(46)
        for t in range(1, cfg["steps"] + 1):
            grads = [g.to(DEV) for g in _config4_grads(shapes, rng, t, cfg["scale_before_step"][t - 1],
                                                       cfg["overflow_steps"])]
            if alternate:
                s = streams[t % 2]
                s.wait_stream(torch.cuda.current_stream(DEV))
                s.wait_stream(streams[(t + 1) % 2])
                opt.step(grads, stream=s)
                for g in grads:
                    g.record_stream(s)
            else:
                opt.step(grads)
        torch.cuda.current_stream(DEV).wait_stream(streams[0])
        torch.cuda.current_stream(DEV).wait_stream(streams[1])
        opt.resolve()
        runs.append((opt, scaler))
    (a, sa), (b, sb) = runs
    assert sa.state_dict() == sb.state_dict() and sb.scale == cfg["final_scale"]
    assert a.skipped_steps == b.skipped_steps == 3
    for p, q in zip(a.param_groups[0]["params"], b.param_groups[0]["params"]):
        assert torch.equal(p, q)
        assert torch.equal(a.state[p]["exp_avg_sq"], b.state[q]["exp_avg_sq"])
        assert a.state[p]["step"] == b.state[q]["step"] == 13


def test_checked_and_detector_steps_interleave(golden_dir):
    """Steps whose flag comes from the producer (checked=True, flag written into
    opt.found_inf) interleaved with steps that run the detector, overflows on both
    kinds: the same bytes, clocks and scale as the step-by-step run."""
    cfg = json.loads((golden_dir / "loss_scale.json").read_text())["config4"]
    shapes = [(384, 200), (777,)]
    masters = [torch.randn(s, generator=torch.Generator().manual_seed(95 + i)) * .02
               for i, s in enumerate(shapes)]
    runs = []
    for sync in (True, False):
        scaler = DynamicLossScale(cfg["initial"], cfg["growth_interval"])
        opt = FusedAdamW([m.to(DEV) for m in masters], lr=3e-4, betas=(.9, .95),
                         weight_decay=.1, loss_scale=scaler, export_dtype=torch.bfloat16, sync=sync)
        rng = np.random.RandomState(47)
        for t in range(1, cfg["steps"] + 1):
            grads = [g.to(DEV) for g in _config4_grads(shapes, rng, t, cfg["scale_before_step"][t - 1],
                                                       cfg["overflow_steps"])]
            if t % 3 == 0:  # the producer tested the gradients
                bad = any(not torch.isfinite(g).all() for g in grads)
                if bad:
                    opt.found_inf.fill_(1)
                opt.step(grads, checked=True)
            else:
                opt.step(grads)
        opt.resolve()
        runs.append((opt, scaler))
    (a, sa), (b, sb) = runs
    assert sa.state_dict() == sb.state_dict() and sb.scale == cfg["final_scale"]
    assert a.skipped_steps == b.skipped_steps == 3 and b.applied_steps == 13
    for p, q in zip(a.param_groups[0]["params"], b.param_groups[0]["params"]):
        assert torch.equal(p, q)
        assert torch.equal(a.state[p]["exp_avg"], b.state[q]["exp_avg"])
    for e, f in zip(a.exports, b.exports):
        assert torch.equal(e, f)


def test_fused_close_with_a_detector_over_several_launches():
    """400 tensors need three detector launches (160 tensors each) and nine AdamW
    launches; the previous step's close rides in exactly one of them.  Eight steps,
    two of them poisoned in the last launch's tensors, end where the step-by-step run ends."""
    gen = torch.Generator().manual_seed(97)
    sizes = [int(torch.randint(1, 3000, (1,), generator=gen)) for _ in range(400)]
    masters = [torch.randn(n, generator=gen) * .02 for n in sizes]
    steps = [[(torch.randn(n, generator=gen) * 1e-3 * 256).half() for n in sizes] for _ in range(8)]
    steps[2][395][0] = float("nan")
    steps[5][399][-1] = float("-inf")
    runs = []
    for sync in (True, False):
        scaler = DynamicLossScale(256.0, growth_interval=3)
        opt = FusedAdamW([m.to(DEV) for m in masters], lr=1e-3, betas=(.9, .95), weight_decay=.1,
                         loss_scale=scaler, sync=sync)
        for gs in steps:
            opt.step([g.to(DEV) for g in gs])
        opt.resolve()
        runs.append((opt, scaler))
    (a, sa), (b, sb) = runs
    assert sa.state_dict() == sb.state_dict()
    assert a.skipped_steps == b.skipped_steps == 2 and b.applied_steps == 6
    for p, q in zip(a.param_groups[0]["params"], b.param_groups[0]["params"]):
        assert torch.equal(p, q)
        assert a.state[p]["step"] == b.state[q]["step"] == 6


@pytest.mark.parametrize("dtype,export,count", [(torch.float32, None, 49), (torch.float16, torch.float16, 401),
                                                (torch.bfloat16, torch.bfloat16, 830)])
def test_descriptor_table_equals_kernel_argument_launches(monkeypatch, dtype, export, count):
    """More than 48 tensors run over the descriptor table in device memory (400 gradients a
    launch), the same bytes as the launches whose descriptors are kernel arguments: sizes at
    the edges of the AdamW and detector blocks, empty ones, views off 16 bytes, two constant
    sets, new gradient buffers, a non-finite value in the first and the last tensor."""
    from morph_amd import kernels
    edges = [0, 1, 3, 255, 256, 257, 4095, 4096, 4097, 8191, 8192, 8193, 20000]
    gen = torch.Generator().manual_seed(count)
    sizes = [edges[i % len(edges)] if i % 3 else int(torch.randint(1, 700, (1,), generator=gen))
             for i in range(count)]
    sizes[0], sizes[-1] = 300, 8193
    place = lambda t, i: torch.cat([torch.zeros(i % 4, dtype=t.dtype), t]).to(DEV)[i % 4:]  # noqa: E731
    masters = [torch.randn(n, generator=gen) * .02 for n in sizes]
    steps = [[(torch.randn(n, generator=gen) * 1e-3 * 64).to(dtype) for n in sizes] for _ in range(4)]
    steps[1][0][299] = float("nan")
    steps[2][-1][8192] = float("inf")
    runs = []
    for table in (True, False):
        if not table:
            monkeypatch.setattr(kernels.AdamwBatch, "_device_table", lambda self: None)
        ps = [place(m, i) for i, m in enumerate(masters)]
        opt = FusedAdamW([dict(params=ps[:7]), dict(params=ps[7:], lr=2e-3, weight_decay=0.0)], lr=1e-3,
                         loss_scale=DynamicLossScale(64.0), export_dtype=export)
        outs = []
        for k, gs in enumerate(steps):
            gs = [place(g, i if k else 0) for i, g in enumerate(gs)]
            assert (opt._cache is None) or (opt._cache[0]._table is not None) == table
            opt.step(gs)
            outs.append([p.clone() for p in ps])
        opt.resolve()
        outs.append([opt.state[p][k] for p in ps for k in ("exp_avg", "exp_avg_sq")] + opt.exports)
        runs.append((opt, outs))
    (a, oa), (b, ob) = runs
    assert a.skipped_steps == b.skipped_steps == 2 and a.applied_steps == b.applied_steps == 2
    for step, (xs, ys) in enumerate(zip(oa, ob)):
        for i, (x, y) in enumerate(zip(xs, ys)):
            assert torch.equal(x, y), (step, i)
    assert not torch.equal(oa[0][0], oa[3][0]) and torch.equal(oa[0][0], oa[2][0])
    strided = torch.zeros(2 * sizes[0], dtype=dtype, device=DEV)[::2]
    with pytest.raises(ValueError, match="contiguous"):
        a.step([strided] + [torch.zeros(n, dtype=dtype, device=DEV) for n in sizes[1:]])


def _group(count, size, seed=5):
    gen = torch.Generator().manual_seed(seed)
    return ([torch.randn(size, generator=gen) * .02 for _ in range(count)],
            [(torch.randn(size, generator=gen) * 1e-3).to(DEV) for _ in range(count)])


@pytest.mark.parametrize("size", [16384, 16385])
def test_large_tensors_get_their_table_when_they_are_stepped_again(monkeypatch, size):
    """Up to 16384 elements a tensor the table is made with the batch; above, at the second step
    of the same tensors, and a loop that alternates between two sets of gradients makes none.
    The same bytes without any."""
    from morph_amd import kernels
    masters, grads = _group(49, size)
    other = [None] + grads[1:-1] + [None]  # 47 tensors: never a table
    fewer = [None] + _group(50, size)[1]
    made, runs = [], []
    for table in (True, False):
        if not table:
            monkeypatch.setattr(kernels.AdamwBatch, "_device_table", lambda self: None)
        ps = [m.to(DEV) for m in masters + masters[:2]]
        opt = FusedAdamW(ps, lr=1e-3)
        for gs in (grads + [None, None], grads + [None, None], other + [None, None],
                   fewer, grads + [None, None], fewer, fewer, fewer):
            opt.step(gs)
            made.append(opt._cache[0]._table is not None)
        opt.resolve()
        runs.append(ps)
    small = size == 16384
    assert made[:8] == [small, True, False, small, small, small, True, True] and not any(made[8:])
    assert all(torch.equal(x, y) for x, y in zip(*runs))


def test_many_tensors_can_be_captured_after_one_step():
    """A step's second time over the same tensors may fall into a graph capture, which allows no
    copy to the device: it goes without a table.  A batch of the kernels module likewise."""
    from morph_amd import kernels
    from morph_amd.hyper import adamw_constants
    masters, grads = _group(49, 20000)
    side = torch.cuda.Stream()
    runs = []
    for captured in (True, False):
        ps = [m.to(DEV) for m in masters]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            opt = FusedAdamW(ps, lr=1e-3)
            opt.step(grads)
            side.synchronize()
            if captured:
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    opt.step(grads)
                    opt.step(grads)
                assert opt._cache[0]._table is None
            for _ in range(3):
                if captured:
                    graph.replay()
                else:
                    opt.step(grads)
                    opt.step(grads)
                side.synchronize()
            opt.resolve()
        runs.append(ps + [opt.state[p]["exp_avg_sq"] for p in ps])
        assert {opt.state[p]["step"] for p in ps} == {7}
    assert all(torch.equal(x, y) for x, y in zip(*runs))

    hp = adamw_constants(lr=1e-3, beta1=.9, beta2=.999, eps=1e-8, weight_decay=.01, step=1)
    runs = []
    for captured in (True, False):
        ps = [m.to(DEV) for m in masters]
        ms, vs = ([torch.zeros_like(p) for p in ps] for _ in range(2))
        torch.cuda.synchronize()
        if captured:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                kernels.AdamwBatch(ps, ms, vs, grads).launch([hp])
        for _ in range(3):
            if captured:
                graph.replay()
            else:
                kernels.AdamwBatch(ps, ms, vs, grads).launch([hp])
            torch.cuda.synchronize()
        runs.append(ps + vs)
    assert all(torch.equal(x, y) for x, y in zip(*runs))


@pytest.mark.parametrize("empty", [range(400, 450), range(0, 400), range(0, 450)],
                         ids=["last launch", "first launch", "all"])
def test_a_table_step_is_stamped_around_its_launches(empty):
    """The start event is stamped by the first launch of a step that has elements, the stop event
    by the last: 450 tensors over the descriptor table, 400 to a launch, those of one empty."""
    from morph_amd import kernels
    n = 1 << 14
    ps = [torch.zeros(0 if i in empty else n, device=DEV) for i in range(450)]
    opt = FusedAdamW(ps, lr=1e-3)
    gs = [torch.ones_like(p) for p in ps]
    opt.step(gs)
    assert opt._cache[0]._table is not None
    opt.dispatch_timer = kernels.DispatchTimer(2)
    opt.step(gs)
    opt.step(gs)
    torch.cuda.synchronize()
    if len(empty) < 450:
        assert all(1e-3 < ms < 50 for ms in opt.dispatch_timer.elapsed_ms())
    assert all(torch.isfinite(p).all() for p in ps)


@pytest.mark.parametrize("count", [5, 60])
def test_native_steps_equal_python_steps(count):
    """From a batch's second step on the launches go out natively (hostpath.cpp).  A sequence that
    takes that path and leaves it -- new buffers, missing gradients, another learning rate,
    checked steps, another stream, overflows, replaced export buffers, a loaded state -- against
    the same sequence kept on the Python path (an optimizer with a launch timer)."""
    gen = torch.Generator().manual_seed(7)
    shapes = [(int(torch.randint(1, 3000, (1,), generator=gen)),) for _ in range(count - 1)] + [(40, 30)]
    masters = [torch.randn(s, generator=gen) * .02 for s in shapes]
    steps = [[(torch.randn(s, generator=gen) * 1e-3 * 1024).half() for s in shapes] for _ in range(14)]
    steps[4][1][0] = float("inf")
    steps[9][-1][3, 3] = float("nan")
    side = torch.cuda.Stream()
    runs, native = [], 0
    for timed in (False, True):
        ps = [m.to(DEV) for m in masters]
        opt = FusedAdamW([dict(params=ps[:2]), dict(params=ps[2:], weight_decay=0.0)], lr=1e-3,
                         loss_scale=DynamicLossScale(1024.0, growth_interval=4), export_dtype=torch.float16)
        for k, gs in enumerate(steps):
            if timed:
                opt.kernel_timer = []
            gs = [g.to(DEV) for g in gs]
            if k in (5, 6):
                gs[2] = None
            if k == 7:
                opt.param_groups[1]["lr"] = 5e-4
            if k == 8:
                opt.set_exports([torch.zeros_like(e) for e in opt.exports])
            if k == 11:
                opt.load_state_dict(copy.deepcopy(opt.state_dict()))
            if k == 12:
                side.wait_stream(torch.cuda.current_stream())
                opt.step(gs, stream=side)
                torch.cuda.current_stream().wait_stream(side)
            else:
                if k == 10:  # flagged by the gradients' producer
                    opt.found_inf.fill_(0)
                opt.step(gs, checked=k == 10)
            native += not timed and opt._cache[2] is None
        opt.resolve()
        runs.append((opt, ps))
    (a, pa), (b, pb) = runs
    assert native == 5  # steps 2, 3, 4, 10 and 13
    assert a.skipped_steps == b.skipped_steps == 2 and a.applied_steps == b.applied_steps
    assert a.loss_scale.state_dict() == b.loss_scale.state_dict()
    for p, q, e, f in zip(pa, pb, a.exports, b.exports):
        assert torch.equal(p, q) and torch.equal(e, f)
        assert torch.equal(a.state[p]["exp_avg_sq"], b.state[q]["exp_avg_sq"])
        assert a.state[p]["step"] == b.state[q]["step"]
    with pytest.raises(ValueError, match="contiguous"):
        a.step([torch.zeros(2 * g.numel(), dtype=torch.half, device=DEV)[::2] for g in gs])


def test_a_failed_launch_closes_the_previous_step_once(monkeypatch):
    """The AdamW launch of a native step fails (the entry point refuses) behind the detector that
    closed the step before it: the error is raised, and the steps that follow count that close
    once and apply as if the failed step had not been asked for."""
    import ctypes

    from morph_amd import _lib
    refuse = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: -1)
    w0 = torch.randn(1000, generator=torch.Generator().manual_seed(3)) * .02
    grads = [torch.randn(1000, generator=torch.Generator().manual_seed(40 + k)).to(DEV) for k in range(5)]
    runs = []
    for fails in (True, False):
        w = w0.to(DEV)
        opt = FusedAdamW([w], lr=1e-3, loss_scale=DynamicLossScale(1024.0))
        for g in grads[:3]:
            opt.step([g])
        if fails:
            real, address = opt._plan, _lib.entry_address
            with monkeypatch.context() as patch:
                patch.setattr(_lib, "entry_address", lambda name: ctypes.cast(
                    refuse, ctypes.c_void_p).value if name == "morph_adamw_multi_dev" else address(name))
                opt._plan = opt._cache[0].step_plan([w], [0], opt._ctl.clocks, opt._ctl.state)
            with pytest.raises(_lib.MorphError):
                opt.step([grads[3]])
            opt._plan = real
        for g in grads[3:]:
            opt.step([g])
        opt.resolve()
        runs.append((w, opt.state[w], opt.applied_steps, opt.loss_scale.state_dict()))
    (w, st, applied, scaler), (rw, rst, rapplied, rscaler) = runs
    assert st["step"] == rst["step"] == 5 and applied == rapplied == 5 and scaler == rscaler
    assert torch.equal(w, rw) and torch.equal(st["exp_avg_sq"], rst["exp_avg_sq"])


@pytest.mark.parametrize("masters_on", ["gpu", "gpu, Python path", "cpu"])
def test_moved_parameters_and_replaced_moments_are_the_ones_stepped(masters_on):
    """Between two steps of the same tensors a caller moves a parameter (p.data, CPU masters too)
    or puts other moments into opt.state: the next step reads and updates what is there now, as
    an optimizer that starts from those values does, and leaves the old storage alone."""
    gen = torch.Generator().manual_seed(23)
    n = 3000
    start = [torch.randn(n, generator=gen) * .02 for _ in range(3)]
    grads = [[torch.randn(n, generator=gen) * 1e-3 for _ in start] for _ in range(8)]
    host = masters_on == "cpu"
    put = (lambda t: t.clone()) if host else (lambda t: t.to(DEV))
    ps = [torch.nn.Parameter(put(t)) for t in start]
    opt = FusedAdamW(ps, lr=1e-3)
    steps = []

    def step(gs):
        if masters_on == "gpu, Python path":
            opt.kernel_timer = []
        opt.step([g.to(DEV) for g in gs])
        steps.append(opt._cache[2] is None)

    ref_w, ref_m, ref_v = ([t.numpy().copy() for t in start], [np.zeros(n, np.float32) for _ in start],
                           [np.zeros(n, np.float32) for _ in start])
    from oracle import reference as R

    def ref(gs, t):
        for i, g in enumerate(gs):
            R.adamw(g.numpy(), ref_w[i], ref_m[i], ref_v[i], R.torch_adamw_hp(1e-3, .9, .999, 1e-8, .01, t))

    t = 0
    for k in range(3):
        t += 1
        step(grads[k]), ref(grads[k], t)
    old = ps[0].data
    opt.resolve()
    was = old.clone()
    moved = torch.randn(n, generator=gen) * .02
    ps[0].data = put(moved)
    ref_w[0] = moved.numpy().copy()
    for k in (3, 4, 5):
        t += 1
        step(grads[k]), ref(grads[k], t)
    opt.resolve()
    assert torch.equal(old, was)
    first, second = torch.randn(n, generator=gen) * 1e-4, torch.rand(n, generator=gen) * 1e-6
    opt.state[ps[1]]["exp_avg"] = first.to(DEV)
    opt.state[ps[2]]["exp_avg_sq"] = second.to(DEV)
    ref_m[1], ref_v[2] = first.numpy().copy(), second.numpy().copy()
    for k in (6, 7):
        t += 1
        step(grads[k]), ref(grads[k], t)
    opt.resolve()
    if masters_on == "gpu":
        assert steps == [False, False, True] * 2 + [False, False]
    else:
        assert not any(steps)
    for i, p in enumerate(ps):
        assert_same_bits(p.detach().cpu().numpy(), ref_w[i], f"master {i}")
        assert_same_bits(opt.state[p]["exp_avg"].cpu().numpy(), ref_m[i], f"exp_avg {i}")
        assert_same_bits(opt.state[p]["exp_avg_sq"].cpu().numpy(), ref_v[i], f"exp_avg_sq {i}")


def test_cpu_masters_need_no_host_extension(monkeypatch, tmp_path):
    """The host extension holds the native step over device masters, and a build of it fits one
    version of torch: without it CPU masters step as with it, and device masters say so."""
    from morph_amd import _lib
    w0 = torch.randn(3000, generator=torch.Generator().manual_seed(5)) * .02
    g = torch.randn(3000, generator=torch.Generator().manual_seed(6))
    with_it, without = w0.clone(), w0.clone()
    opt = FusedAdamW([with_it], lr=1e-3)
    for _ in range(3):
        opt.step([g])
    monkeypatch.setattr(_lib, "_hostpath", None)
    monkeypatch.setattr(_lib, "HOSTPATH_PATH", tmp_path / "_hostpath.so")
    opt = FusedAdamW([without], lr=1e-3)
    for _ in range(3):
        opt.step([g])
    assert torch.equal(with_it, without) and not torch.equal(without, w0)
    with pytest.raises(ImportError):
        FusedAdamW([w0.to(DEV)])


class _Sub(torch.nn.Parameter):
    pass


@pytest.mark.parametrize("how", ["subclass", "dispatch mode"])
def test_parameters_the_native_path_cannot_describe_step_as_others(how):
    """Parameters of a tensor subclass, and steps under a TorchDispatchMode (a FLOP counter,
    say), take the Python path on every step, with the bits of plain parameters' steps."""
    import contextlib

    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    gen = torch.Generator().manual_seed(17)
    masters = [torch.randn(n, generator=gen) * .02 for n in (300, 70)]
    grads = [[torch.randn(n, generator=gen) * 1e-3 for n in (300, 70)] for _ in range(4)]
    runs = []
    for odd in (True, False):
        sub = odd and how == "subclass"
        ps = [m.to(DEV).as_subclass(_Sub) if sub else torch.nn.Parameter(m.to(DEV)) for m in masters]
        opt = FusedAdamW(ps, lr=1e-3)
        for gs in grads:
            for p, g in zip(ps, gs):
                p.grad = g.to(DEV)
            with Mode() if odd and not sub else contextlib.nullcontext():
                opt.step()
        opt.resolve()
        runs.append([p.detach().as_subclass(torch.Tensor) for p in ps])
    for x, y, m in zip(*runs, masters):
        assert torch.equal(x, y) and not torch.equal(x.cpu(), m)


@pytest.mark.parametrize("count,size", [(1, 1 << 24), (200, 1 << 16)], ids=["one", "split"])
def test_dispatch_timer_stamps_the_adamw_launches(count, size):
    """Events stamped by the AdamW dispatch itself (hipExtLaunchKernel) time the pass: each
    interval lies inside the events recorded around the launch (which may also hold host
    delays) and is no shorter than the HBM traffic of the FP32 state at the 8 TB/s peak
    (24 B/param: master and moments read and written); a call split into several launches
    (200 tensors) runs from the first start to the last end."""
    from morph_amd.kernels import DispatchTimer
    gen = torch.Generator(device=DEV).manual_seed(98)
    ps = [torch.randn(size, generator=gen, device=DEV) * .02 for _ in range(count)]
    gs = [torch.randn(size, generator=gen, device=DEV).half() for _ in range(count)]
    opt = FusedAdamW(ps, lr=1e-3)
    opt.step(gs)
    opt.dispatch_timer = DispatchTimer(4, DEV)
    opt.kernel_timer = []
    for _ in range(4):
        opt.step(gs)
    torch.cuda.synchronize()
    stamped = opt.dispatch_timer.elapsed_ms()
    around = [a.elapsed_time(b) for a, b in opt.kernel_timer]
    assert len(stamped) == 4
    floor_ms = 24 * count * size / 8e12 * 1e3
    for x, y in zip(stamped, around):
        assert floor_ms <= x <= y + 0.002, (x, y, floor_ms)
    with pytest.raises(RuntimeError):
        opt.step(gs)  # the timer holds four pairs
    opt.dispatch_timer = None
    opt.resolve()
    assert opt.applied_steps == 5

def _config4_grads(shapes, rng, t, scale, overflow_steps):
    grads = bench.config2_grads("cpu", 2000 + t, shapes, scale=scale)
    if t in overflow_steps:
        for _ in range(int(rng.randint(1, 9))):
            k = int(rng.randint(len(grads)))
            flat = grads[k].view(-1)
            flat[int(rng.randint(flat.numel()))] = float(rng.choice([np.inf, -np.inf, np.nan]))
    return grads


def test_async_steps_equal_synchronous_steps(golden_dir):
    """16 steps enqueued back to back (no host round trip) end in the same bytes, clocks
    and loss scale as the step-by-step run, though the host learns the outcomes only at
    the end.  Gradients are pre-scaled with the scale sequence the skips imply."""
    cfg = json.loads((golden_dir / "loss_scale.json").read_text())["config4"]
    shapes = [(512, 256), (256, 512), (1000,)]
    masters = [torch.randn(s, generator=torch.Generator().manual_seed(60 + i)) * .02
               for i, s in enumerate(shapes)]
    runs = []
    for sync in (True, False):
        scaler = DynamicLossScale(cfg["initial"], cfg["growth_interval"])
        opt = FusedAdamW([m.to(DEV) for m in masters], lr=3e-4, betas=(.9, .95),
                         weight_decay=.1, loss_scale=scaler, export_dtype=torch.float16, sync=sync)
        rng = np.random.RandomState(45)
        for t in range(1, cfg["steps"] + 1):
            grads = _config4_grads(shapes, rng, t, cfg["scale_before_step"][t - 1],
                                   cfg["overflow_steps"])
            opt.step([g.to(DEV) for g in grads])
        opt.resolve()
        runs.append((opt, scaler))
    (a, sa), (b, sb) = runs
    assert sa.state_dict() == sb.state_dict() and sa.scale == cfg["final_scale"]
    assert a.skipped_steps == b.skipped_steps == 3 and a.applied_steps == b.applied_steps == 13
    for p, q in zip(a.param_groups[0]["params"], b.param_groups[0]["params"]):
        assert torch.equal(p, q)
        for k in ("exp_avg", "exp_avg_sq"):
            assert torch.equal(a.state[p][k], b.state[q][k])
        assert a.state[p]["step"] == b.state[q]["step"] == 13
    for e, f in zip(a.exports, b.exports):
        assert torch.equal(e, f)


def test_overflow_at_minimum_scale_raises_and_freezes_state():
    """precision.py:9-10: overflow at scale <= 1 raises with the state unchanged; on the
    device every step after it is a no-op until the host sees the error."""
    w = torch.randn(4096, generator=torch.Generator().manual_seed(3)).to(DEV)
    scaler = DynamicLossScale(2., growth_interval=2000)
    opt = FusedAdamW([w], lr=1e-3, loss_scale=scaler)
    good = torch.randn(4096, device=DEV).half()
    bad = good.clone()
    bad[5] = float("inf")
    opt.step([good])
    opt.step([bad])   # scale 2 -> 1
    opt.step([bad])   # at scale 1: the reference raises here
    before = w.clone()
    opt.step([good])  # enqueued before the host knows: must change nothing
    with pytest.raises(FloatingPointError, match="minimum loss scale"):
        opt.resolve()
    assert torch.equal(w, before)
    assert scaler.scale == 1.0 and opt.state[w]["step"] == 1


def test_fixed_scale_and_raise_policy():
    """A float loss scale never changes; on_overflow='raise' raises before any mutation."""
    w = torch.randn(3000, generator=torch.Generator().manual_seed(4)).to(DEV)
    opt = FusedAdamW([w], lr=1e-3, loss_scale=1024.0, on_overflow="raise")
    g = (torch.randn(3000, device=DEV) * 1e-3 * 1024).half()
    assert opt.step([g]) is True
    before = w.clone()
    g[0] = float("nan")
    with pytest.raises(FloatingPointError, match="nonfinite gradient"):
        opt.step([g])
    assert torch.equal(w, before) and opt.state[w]["step"] == 1
    g[0] = 0.0
    assert opt.step([g]) is True and opt.state[w]["step"] == 2


def test_loss_scale_growth_on_device_matches_host_rule():
    """growth_interval 3: the scale doubles every 3 clean steps, capped at 65536."""
    from oracle import reference as R
    w = torch.randn(2048, generator=torch.Generator().manual_seed(5)).to(DEV)
    scaler = DynamicLossScale(16384., growth_interval=3)
    oscaler = R.LossScale(16384., 3)
    opt = FusedAdamW([w], lr=1e-3, loss_scale=scaler)
    for t in range(14):
        opt.step([(torch.randn(2048, device=DEV) * 1e-4).half()])
        oscaler.success()
    opt.resolve()
    assert scaler.state_dict() == oscaler.state_dict() and scaler.scale == 65536.


@pytest.mark.parametrize("mode", ["host_scale", "device_scale"])
def test_loss_scaled_by_the_exposed_scale_across_overflow_and_growth(mode):
    """A training loop scales each step's loss by the scale the API exposes -- the host
    DynamicLossScale's `scale` (which settles the queued steps when read) or the
    optimizer's device scale (scale_loss / loss_scale_tensor, no wait) -- and never
    calls resolve().  With growth every 3 clean steps and overflows at steps 4 and 9
    the scale moves 1024 -> 2048 -> 1024 -> 2048 -> 1024 ..., and every applied step
    must unscale by exactly the factor its gradient was scaled with: bit-exact
    against the oracle running the reference's loop (disk.py:483-496)."""
    from oracle import reference as R
    n = 5000
    w0 = torch.randn(n, generator=torch.Generator().manual_seed(31)) * .02
    scaler = DynamicLossScale(1024., growth_interval=3)
    w = w0.to(DEV)
    opt = FusedAdamW([w], lr=3e-4, betas=(.9, .95), weight_decay=.1, loss_scale=scaler)
    gen = torch.Generator().manual_seed(32)
    true_grads = [torch.randn(n, generator=gen) * 1e-4 for _ in range(12)]
    ow, om, ov = w0.numpy().copy(), np.zeros(n, np.float32), np.zeros(n, np.float32)
    oscaler, ot, seen = R.LossScale(1024., 3), 0, []
    for k, g in enumerate(true_grads):
        if mode == "host_scale":
            scale = scaler.scale                     # the reference reads scaler.scale
            g16 = (g * scale).half().to(DEV)         # backward of loss * scale
        else:
            g16 = opt.scale_loss(g.to(DEV)).half()   # the same product on the GPU
        if k + 1 in (4, 9):
            g16[17] = float("inf")
        opt.step([g16])
        seen.append(oscaler.scale)
        o16 = (g * oscaler.scale).half()
        if k + 1 in (4, 9):
            oscaler.overflow()
            continue
        ot += 1
        R.adamw(o16.numpy(), ow, om, ov,
                R.torch_adamw_hp(3e-4, .9, .95, 1e-8, .1, ot, scale=oscaler.scale))
        oscaler.success()
    assert seen[:10] == [1024.] * 3 + [2048., 1024., 1024., 1024., 2048., 2048., 1024.]
    assert scaler.scale == oscaler.scale and scaler.good_steps == oscaler.good_steps
    assert_same_bits(w.cpu().numpy(), ow, "master")
    assert_same_bits(opt.state[w]["exp_avg"].cpu().numpy(), om, "exp_avg")
    assert opt.state[w]["step"] == ot == 10


@pytest.mark.parametrize("how", ["assign", "load_state_dict"])
def test_caller_edits_of_the_scaler_reach_the_device(how):
    """disk.py:245/509 and single_pass.py:183-184 restore the scaler on resume: a scale
    set on the host between steps (while earlier steps are still queued) is the scale
    the next step unscales by, bit-exact against the oracle, and the host keeps it."""
    from oracle import reference as R
    n = 3000
    w0 = torch.randn(n, generator=torch.Generator().manual_seed(36)) * .02
    w = w0.to(DEV)
    scaler = DynamicLossScale(65536., growth_interval=2000)
    opt = FusedAdamW([w], lr=3e-4, betas=(.9, .95), weight_decay=.1, loss_scale=scaler)
    gen = torch.Generator().manual_seed(37)
    grads = [torch.randn(n, generator=gen) * 1e-4 for _ in range(4)]
    ow, om, ov = w0.numpy().copy(), np.zeros(n, np.float32), np.zeros(n, np.float32)
    for t in (1, 2):  # queued, not resolved
        g16 = (grads[t - 1] * 65536.).half()
        opt.step([g16.to(DEV)])
        R.adamw(g16.numpy(), ow, om, ov, R.torch_adamw_hp(3e-4, .9, .95, 1e-8, .1, t, scale=65536.))
    if how == "assign":
        scaler.scale = 1024.
        expect_good = 2          # the queued steps' successes stand
    else:
        scaler.load_state_dict({"scale": 1024., "good_steps": 7, "growth_interval": 2000})
        expect_good = 7
    assert scaler.scale == 1024.
    for t in (3, 4):
        g16 = (grads[t - 1] * 1024.).half()
        opt.step([g16.to(DEV)])
        R.adamw(g16.numpy(), ow, om, ov, R.torch_adamw_hp(3e-4, .9, .95, 1e-8, .1, t, scale=1024.))
    opt.resolve()
    assert opt.loss_scale_tensor().item() == 1024.
    assert scaler.scale == 1024. and scaler.good_steps == expect_good + 2
    assert_same_bits(w.cpu().numpy(), ow, "master")
    assert_same_bits(opt.state[w]["exp_avg_sq"].cpu().numpy(), ov, "exp_avg_sq")


def test_after_the_minimum_scale_raise_the_optimizer_goes_on():
    """precision.py:9-11 raises and leaves the scaler usable: after the raise is reported
    (once), state_dict() works, load_state_dict() restores, and the next step applies."""
    w = torch.randn(4096, generator=torch.Generator().manual_seed(33)).to(DEV)
    scaler = DynamicLossScale(1., growth_interval=2000)
    opt = FusedAdamW([w], lr=1e-3, loss_scale=scaler)
    good = torch.randn(4096, device=DEV).half()
    bad = good.clone()
    bad[9] = float("nan")
    opt.step([good])
    saved = opt.state_dict()
    saved = {"state": {k: {kk: vv.clone() for kk, vv in v.items()} for k, v in saved["state"].items()},
             "param_groups": saved["param_groups"]}
    w_saved = w.clone()
    opt.step([bad])                      # overflow at scale 1: the reference raises here
    snapshot = opt.state_dict()          # reading the state does not raise
    assert snapshot["state"][0]["step"].item() == 1.0
    with pytest.raises(FloatingPointError, match="minimum loss scale"):
        opt.resolve()
    opt.resolve()                        # reported once
    opt.step([good])                     # and the optimizer goes on
    opt.resolve()
    assert opt.state[w]["step"] == 2 and scaler.scale == 1.0
    # fatal again, then restore a saved state: the restored optimizer steps normally
    opt.step([bad])
    w.copy_(w_saved)
    opt.load_state_dict(saved)
    opt.step([good])
    opt.resolve()
    assert opt.state[w]["step"] == 2


def test_memory_read_under_another_current_stream_is_noted(monkeypatch):
    """An optimizer's clock list and bias tables are allocated on the stream that is current at
    its first step; steps under another current stream read them there, so the allocator is
    told: a list replaced by another set of gradients is not handed out under that work."""
    noted = []
    real = torch.Tensor.record_stream
    monkeypatch.setattr(torch.Tensor, "record_stream",
                        lambda t, s: (noted.append((t.data_ptr(), s)), real(t, s))[1])
    ps = [torch.zeros(100, device=DEV) for _ in range(2)]
    gs = [torch.ones(100, device=DEV) for _ in range(2)]
    opt = FusedAdamW(ps, lr=1e-3)
    opt.step(gs)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            opt.step(gs)
    clock_list, table = opt._cache[1], opt._tables[(.9, .999)]
    assert (clock_list.data_ptr(), side) in noted and side in table._streams
    old = (table.bc1.data_ptr(), side)
    opt._bound = 4096
    with torch.cuda.stream(side):
        opt.step(gs)
    assert old in noted and side in table._streams
    opt.resolve()


def test_bias_tables_grow_past_4096_steps_on_a_side_stream():
    """The bias-correction tables double at step 4097; the old ones stay valid for the
    side stream's queued launches.  Result bit-exact against the oracle."""
    from oracle import reference as R
    n = 1000
    w0 = torch.randn(n, generator=torch.Generator().manual_seed(34)) * .02
    w = w0.to(DEV)
    opt = FusedAdamW([w], lr=1e-4, betas=(.9, .95), weight_decay=.1)
    g = (torch.randn(n, generator=torch.Generator().manual_seed(35)) * 1e-3)
    gd = g.to(DEV)
    side = torch.cuda.Stream(DEV)
    side.wait_stream(torch.cuda.current_stream(DEV))
    steps = 4100
    for _ in range(steps):
        opt.step([gd], stream=side)
    opt.resolve()
    torch.cuda.synchronize()
    ow, om, ov = w0.numpy().copy(), np.zeros(n, np.float32), np.zeros(n, np.float32)
    for t in range(1, steps + 1):
        R.adamw(g.numpy(), ow, om, ov, R.torch_adamw_hp(1e-4, .9, .95, 1e-8, .1, t))
    assert opt.state[w]["step"] == steps
    assert_same_bits(w.cpu().numpy(), ow, "master")
    assert_same_bits(opt.state[w]["exp_avg_sq"].cpu().numpy(), ov, "exp_avg_sq")
