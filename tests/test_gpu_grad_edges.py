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
