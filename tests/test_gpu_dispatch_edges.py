"""Branches of the evaluator's and the gradient's dispatch that only many tapes reach, and Langevin
blocks on programs that fill their cap."""
import numpy as np
import pytest

from gpu_util import check_paths, dev, kappas, ll_agree, say
from test_gpu_interpreter import batch, dataset

pytestmark = pytest.mark.gpu


def tiled(tensors, count):
    """Device arrays [.., k] repeated along their last axis to `count` columns, on the device."""
    import torch
    k = tensors[0].shape[-1]
    idx = torch.arange(count, device="cuda") % k
    return [t.index_select(t.dim() - 1, idx).contiguous() for t in tensors]


@pytest.mark.parametrize("n", [40, 100, 300])
@pytest.mark.parametrize("tapes", [2049, 40961, 61447, 81923])
def test_several_tapes_per_wave(oracle, gpr, tapes, n):
    """From 40960 tapes on a wave takes two to four, the next loaded while one is evaluated; the
    counts leave a last wave and a last workgroup short.  One, two and four points per lane: the
    bits of the same tapes evaluated as a small batch."""
    import torch
    cap = 128
    O, V, L = batch(oracle, cap)
    k = O.shape[1]
    small = [dev(O), dev(V), dev(L)]
    many = tiled(small, tapes)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(n, uneven=True)], [1])
        torch.cuda.synchronize()
        say(f"{tapes} tapes at n={n}")
        out = []
        for o, v, ln in (small, many):
            ll = torch.full((ln.shape[0],), 7.0, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            ctx.eval_loglik_dev(0, o.data_ptr(), v.data_ptr(), ln.data_ptr(), ln.shape[0], cap, gpr.SCHED_WAVE, ll.data_ptr())
            out.append(ll)
    assert bool(torch.isfinite(out[0]).all())
    assert torch.equal(tiled([out[0]], tapes)[0], out[1])


@pytest.mark.parametrize("cap,n", [(64, 40), (128, 200), (128, 300), (64, 1025)])
def test_gradients_of_many_tapes(oracle, gpr, cap, n):
    """Above 2048 tapes the gradient loads only the rows below a tape's length: the bits of the same
    tapes as a small batch (sizes whose workgroups are the same on both sides)."""
    import torch
    O, V, L = batch(oracle, cap)
    small = [dev(O), dev(V), dev(L)]
    tapes = 2049
    many = tiled(small, tapes)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(n, uneven=False)], [1])
        torch.cuda.synchronize()
        say(f"gradients of {tapes} tapes, cap {cap}, n={n}")
        out = []
        for o, v, ln in (small, many):
            g = torch.full_like(v, 7.0)
            lp = torch.full((ln.shape[0],), 7.0, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            ctx.grad_logpost_dev(0, o.data_ptr(), v.data_ptr(), ln.data_ptr(), ln.shape[0], cap, g.data_ptr(), lp.data_ptr())
            out.append((g, lp))
    g, lp = tiled([*out[0]], tapes)
    assert torch.equal(g, out[1][0]) and torch.equal(lp, out[1][1])


@pytest.mark.parametrize("cap", [64, 128])
def test_mala_on_full_programs_holds_its_state(oracle, gpr, cap):
    """Langevin moves on programs of 62 to cap tokens: after the block a chain's prior is its
    program's bit for bit and its likelihood the oracle's, and a chain away from the oracle's (by
    1e-3, the device sums gradients in FP32) met an accept decision within 1e-4 of the likelihood's
    scale: twice 1e-5 for the likelihoods and as much for the drift terms, with a margin."""
    O, V, L = batch(oracle, cap)
    keep = np.flatnonzero((L >= 60) | (L <= 13))
    O, V, L = O[:, keep].copy(), V[:, keep].copy(), L[keep].copy()
    x, y, sd = dataset(150, uneven=True)
    steps, nch = 24, len(L)
    cfg = oracle.make_cfg(cap=cap, seed=5, fixed_structure=1, proposal=1, eps=0.01, sigma=0.05)
    o_ops, o_cs, o_ln = O.copy(), V.copy(), L.copy()
    m = np.zeros(nch)
    oracle.cfg_run_block(cfg, o_ops, o_cs, o_ln, x, y, sd, 0, steps, margin=m)
    with gpr.Context(cap=cap, seed=5, fixed_structure=1, proposal=gpr.PROP_MALA, eps=0.01, sigma=0.05,
                     schedule=gpr.SCHED_WAVE, resample=gpr.RS_NONE) as ctx:
        ctx.set_data([(x, y, sd)], [nch])
        ctx.write_state(O, V, L)
        say(f"mala on full programs cap={cap}")
        ctx.run_block(steps)
        ops, cs, ln, pr, ll = ctx.read_state()
        st = ctx.stats()
    assert st.const_accepted > 0 and np.array_equal(ops, O) and np.array_equal(ln, L)
    assert np.array_equal(pr, [oracle.tape_prior(ops[:ln[i], i], cs[:ln[i], i], 10) for i in range(nch)])
    ref = np.array([oracle.tape_loglik(ops[:ln[i], i], cs[:ln[i], i], x, y, sd, mode=2) for i in range(nch)])
    kap = kappas(oracle, ops, cs, ln, range(nch), x, y, sd)
    ok, _ = ll_agree(ll, ref, len(x), kap, sd)
    assert ok.all(), np.flatnonzero(~ok)
    close = np.all(np.abs(cs - o_cs) <= 1e-3 * np.maximum(1.0, np.abs(o_cs)), axis=0)
    check_paths(close, m, f"mala on full programs cap={cap}:", rel=1e-4)
