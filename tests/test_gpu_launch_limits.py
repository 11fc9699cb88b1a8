"""Calls of more tapes than one launch has room for: a launch holds fewer than 2^32 threads, and
the kernels with a workgroup per tape take 64 to 512 of them a tape."""
import numpy as np
import pytest

from gpu_util import say
from test_gpu_interpreter import dataset

pytestmark = pytest.mark.gpu


def one_token_tapes(gpr, n):
    """n tapes of one token, a constant each: small enough to hold millions of them."""
    import torch
    ops = torch.full((1, n), gpr.OP["CONST"], dtype=torch.uint8, device="cuda")
    cs = (torch.arange(n, device="cuda") % 1021).to(torch.float32)[None, :].contiguous() / 1021
    return ops, cs, torch.ones(n, dtype=torch.int32, device="cuda")


def same_by_constant(v):
    """Equal constants have equal results wherever their tapes lie: the first 1021 repeated."""
    import torch
    n = v.shape[0]
    whole = n // 1021 * 1021
    return bool((v[:whole].view(-1, 1021) == v[:1021]).all()) and torch.equal(v[whole:], v[:n - whole])


@pytest.mark.parametrize("tapes,n", [((1 << 23) + 3, 513), ((1 << 25) + 3, 130)])
def test_gradients_of_more_tapes_than_one_launch(gpr, tapes, n):
    import torch
    ops, cs, ln = one_token_tapes(gpr, tapes)
    grad, lp = torch.full_like(cs, 7.0), torch.full((tapes,), 7.0, dtype=torch.float64, device="cuda")
    x, y, sd = dataset(n, uneven=False)
    with gpr.Context(cap=1) as ctx:
        ctx.set_data([(x, y, sd)], [1])
        torch.cuda.synchronize()
        say(f"gradients of {tapes} tapes at n={n}")
        ctx.grad_logpost_dev(0, ops.data_ptr(), cs.data_ptr(), ln.data_ptr(), tapes, 1, grad.data_ptr(), lp.data_ptr())
    c = cs[0, :1021].cpu().numpy().astype(np.float64)
    want = 4.0 * (y.astype(np.float64).sum() - n * c) - 2.0 * c / (1.0 + c * c)       # sd = 0.5: d/dc of -2 sum (c - y)^2
    got = grad[0, :1021].cpu().numpy()
    assert np.max(np.abs(got - want)) <= 1e-4 * np.max(np.abs(want))
    assert same_by_constant(grad[0]) and same_by_constant(lp)


def test_likelihoods_of_more_tapes_than_one_launch(gpr):
    import torch
    tapes, n = (1 << 24) + 3, 513
    ops, cs, ln = one_token_tapes(gpr, tapes)
    x, y, sd = dataset(n, uneven=False)
    ll, ll2 = (torch.full((tapes,), 7.0, dtype=torch.float64, device="cuda") for _ in range(2))
    with gpr.Context(cap=1) as ctx:
        ctx.set_data([(x, y, sd)], [1])
        torch.cuda.synchronize()
        say(f"likelihoods of {tapes} tapes at n={n}")
        ctx.eval_loglik_dev(0, ops.data_ptr(), cs.data_ptr(), ln.data_ptr(), tapes, 1, gpr.SCHED_WAVE, ll.data_ptr())
    dx, dy, dsd = (torch.from_numpy(v).cuda() for v in (x, y, sd))
    torch.cuda.synchronize()
    gpr.eval_loglik_noalloc_async(0, dx.data_ptr(), dy.data_ptr(), dsd.data_ptr(), n, ops.data_ptr(), cs.data_ptr(),
                                  ln.data_ptr(), tapes, 1, gpr.SCHED_WAVE, ll2.data_ptr(),
                                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    c = cs[0, :1021].cpu().numpy().astype(np.float64)
    want = -n * np.log(0.5 * np.sqrt(2 * np.pi)) - 2.0 * np.sum((c[:, None] - y.astype(np.float64)) ** 2, axis=1)
    for v in (ll, ll2):
        assert np.max(np.abs(v[:1021].cpu().numpy() - want) / np.maximum(np.abs(want), n)) <= 1e-5
        assert same_by_constant(v)
