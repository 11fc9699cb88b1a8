"""gpr_grad_logpost where the split of its work changes: datasets around the chunks, the
waves of a workgroup and the rounds of 1024 points, programs from one token to the cap (one
row to more than every wave has), few tapes and many."""
import numpy as np
import pytest

from gpu_util import dev, say
from test_gpu_interpreter import batch, dataset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,n,copies", [(64, 1, 1), (128, 64, 1), (64, 65, 1), (128, 128, 1), (128, 129, 1), (64, 256, 1),
                                          (128, 257, 1), (64, 512, 1), (64, 513, 1), (128, 1024, 1), (128, 1025, 1),
                                          (64, 2100, 1), (128, 1025, 30)])
def test_gradients_at_the_edges(oracle, gpr, cap, n, copies):
    import torch
    O, V, L = batch(oracle, cap)
    k = O.shape[1]
    O, V, L = np.tile(O, (1, copies)), np.tile(V, (1, copies)), np.tile(L, copies)
    x, y, sd = dataset(n, uneven=n % 2 == 1)
    N = O.shape[1]
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([(x, y, sd)], [1])
        dO, dV, dL = dev(O), dev(V), dev(L)
        g = torch.full((cap, N), 7.0, dtype=torch.float32, device="cuda")
        lp = torch.zeros(N, dtype=torch.float64, device="cuda")
        ll = torch.zeros(N, dtype=torch.float64, device="cuda")
        say(f"gradient edges cap={cap} n={n} tapes={N}")
        ctx.grad_logpost_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), N, cap, g.data_ptr(), lp.data_ptr())
        ctx.eval_loglik_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), N, cap, gpr.SCHED_WAVE, ll.data_ptr())
        g, lp, ll = g.cpu().numpy(), lp.cpu().numpy(), ll.cpu().numpy()
    for i in range(k):
        o, v = O[:L[i], i], V[:L[i], i]
        assert lp[i] == oracle.tape_prior(o, v, 10) + ll[i]
        rc, g64, _ = oracle.tape_grad(o, v, x, y, sd)
        assert rc == 0
        scale = max(np.max(np.abs(g64)), 1e-30)
        assert np.max(np.abs(g[:L[i], i] - g64)) <= 1e-4 * scale, (i, int(L[i]))
        assert not g[L[i]:, i].any()
    for c in range(1, copies):      # a tape's result does not depend on its place
        assert np.array_equal(g[:, :k], g[:, c * k:(c + 1) * k]) and np.array_equal(lp[:k], lp[c * k:(c + 1) * k])


@pytest.mark.parametrize("fault", ["none", "zero length", "length over cap", "op past the end", "pops an empty stack",
                                   "two values left", "depth 17"])
@pytest.mark.parametrize("cap", [40, 100])
def test_tapes_checked_on_the_device(oracle, gpr, cap, fault):
    """gpr_grad_logpost_checked reports what the host check of the same tapes reports, and the
    torch function raises its message, with one bad tape among many."""
    import torch
    from gpuropolis_amd import autograd
    n = 130
    O = np.zeros((cap, n), dtype=np.uint8)
    L = np.full(n, 5, dtype=np.int64)
    x, c, add, mul = (gpr.OP[k] for k in ("X", "CONST", "ADD", "MUL"))
    O[:5] = np.array([c, x, mul, c, add], dtype=np.uint8)[:, None]
    bad = 77
    if fault == "zero length":
        L[bad] = 0
    elif fault == "length over cap":
        L[bad] = cap + 1
    elif fault == "op past the end":
        O[cap - 1, bad] = len(gpr.OPS)
    elif fault == "pops an empty stack":
        O[:5, bad] = [x, add, x, x, add]
    elif fault == "two values left":
        L[bad] = 4
    elif fault == "depth 17":
        O[:33, bad] = [x] * 17 + [add] * 16
        L[bad] = 33
    want = None
    try:
        autograd.check_tapes(torch.from_numpy(O), torch.from_numpy(L))
    except gpr.GprError as e:
        want = str(e)
    assert (want is None) == (fault == "none")
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(70, False)], [1])
        say(f"device check: {fault}, cap {cap}")
        for dtype in (torch.int32, torch.int64):
            cs = torch.full((cap, n), 0.5, device="cuda", requires_grad=True)
            args = (ctx, 0, dev(O), cs, dev(L).to(dtype))
            if want is None:
                autograd.log_posterior(*args).sum().backward()
                assert bool(torch.isfinite(cs.grad).all())
            else:
                with pytest.raises(gpr.GprError) as e:
                    autograd.log_posterior(*args)
                assert str(e.value) == want
