"""The wave interpreter at the edges of its registers and rows: tapes that end, or hold a
fused leaf and operator, around tokens 62-64 and 127, stacks at the depths where the
evaluator changes its points per lane, datasets around its chunks, and MH blocks on
programs that fill their cap."""
import numpy as np
import pytest

from gpu_util import check_paths, dev, say

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 5, 61, 62, 63, 64, 65, 66, 67, 126, 127, 128]
DEPTHS = [2, 5, 6, 7, 9, 10, 15, 16]


def chain_tape(length, shift):
    """x, then leaf/operator pairs; `shift` negations in front move the pairs by a token, and
    negations at the end (a handler without a second token) fill an even length."""
    toks = ["X"] + ["NEG"] * min(shift, length - 1)
    k = 0
    while len(toks) + 2 <= length:
        leaf, op = [(("CONST", 0.5), "ADD"), ("X", "MUL"), (("CONST", 0.75), "MUL"), ("X", "SUB"), ("X", "ADD"),
                    (("CONST", 0.25), "SUB")][k % 6]
        toks += [leaf, op]
        k += 1
    return toks + ["NEG"] * (length - len(toks))


def deep_tape(depth):
    """`depth` leaves, then the operators: every push and pop of the stack's rows."""
    leaves = [("CONST", 0.5) if k % 2 else "X" for k in range(depth)]
    return leaves + [("ADD", "MUL", "SUB")[k % 3] for k in range(depth - 1)]


def batch(oracle, cap):
    tapes = [chain_tape(n, s) for n in LENGTHS if n <= cap for s in (0, 1)] + [deep_tape(d) for d in DEPTHS if 2 * d <= cap]
    # a token without a handler between the others, also as the last of a half tape
    tapes += [chain_tape(n, 0)[:-1] + ["EXP"] for n in (62, 64, 66, 126) if n <= cap]
    tapes += [["X", ("CONST", 3.0), "ADD", "EXP", "X", "X", "MUL", ("CONST", 2.0), "ADD", "DIV", "NEG", "X", "SUB"]]
    arrs = [oracle.tape_arrays(t) for t in tapes]
    O = np.zeros((cap, len(arrs)), dtype=np.uint8)
    V = np.zeros((cap, len(arrs)), dtype=np.float32)
    for i, (o, v) in enumerate(arrs):
        O[:len(o), i] = o
        V[:len(o), i] = v
    return O, V, np.array([len(o) for o, _ in arrs], dtype=np.int32)


def dataset(n, uneven):
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, n)
    sd = rng.uniform(0.5, 1.0, n) if uneven else np.full(n, 0.5)
    return x.astype(np.float32), (x + rng.normal(0, 0.5, n)).astype(np.float32), sd.astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 256, 257, 513, 1024, 1025, 2100])
@pytest.mark.parametrize("cap", [64, 128])
def test_eval_at_the_edges(oracle, gpr, n, cap):
    """Every operation of these tapes is exactly rounded on both sides and the sums differ in
    order only: 1e-6 of max(|LL|, n), against FP32 sums of n terms in the oracle's order."""
    import torch
    O, V, L = batch(oracle, cap)
    d = dataset(n, uneven=n % 2 == 1)
    N = O.shape[1]
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([d], [1])
        out = torch.zeros(N, dtype=torch.float64, device="cuda")
        say(f"interpreter edges n={n} cap={cap} tapes={N}")
        dO, dV, dL = dev(O), dev(V), dev(L)
        ctx.eval_loglik_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), N, cap, gpr.SCHED_WAVE, out.data_ptr())
        got = out.cpu().numpy()
    ref = np.array([oracle.tape_loglik(O[:L[i], i], V[:L[i], i], *d) for i in range(N)])
    assert np.all(np.isfinite(ref))
    exp = np.array([gpr.OP["EXP"] in O[:L[i], i] for i in range(N)])
    tol = np.where(exp, 1e-5, 1e-6) * np.maximum(np.abs(ref), n)      # exp: the device's libm
    assert np.all(np.abs(got - ref) <= tol), np.flatnonzero(np.abs(got - ref) > tol)


@pytest.mark.parametrize("cap,n,mala", [(64, 20, 0), (64, 40, 0), (64, 150, 0), (128, 20, 0), (128, 150, 0), (64, 150, 1),
                                        (128, 150, 1)])
def test_blocks_on_full_programs(oracle, gpr, cap, n, mala):
    """Constant steps on programs of 62 to cap tokens (all sizes of one register, and of two),
    one point per lane and with speculative steps (n <= 32): the oracle's trajectories."""
    O, V, L = batch(oracle, cap)
    keep = np.flatnonzero((L >= 60) | (L <= 13))
    O, V, L = O[:, keep].copy(), V[:, keep].copy(), L[keep].copy()
    x, y, sd = dataset(n, uneven=True)
    steps, nch = 24, len(L)
    cfg = oracle.make_cfg(cap=cap, seed=5, fixed_structure=1, proposal=mala, eps=0.01, sigma=0.05)
    o_ops, o_cs, o_ln = O.copy(), V.copy(), L.copy()
    m = np.zeros(nch)
    p_ref, _, _ = oracle.cfg_run_block(cfg, o_ops, o_cs, o_ln, x, y, sd, 0, steps, margin=m)
    with gpr.Context(cap=cap, seed=5, fixed_structure=1, proposal=mala, eps=0.01, sigma=0.05,
                     schedule=gpr.SCHED_WAVE) as ctx:
        ctx.set_data([(x, y, sd)], [nch])
        ctx.write_state(O, V, L)
        say(f"blocks on full programs cap={cap} n={n} mala={mala}")
        ctx.run_block(steps)
        g_ops, g_cs, g_ln, g_pr, _ = ctx.read_state()
    if mala:      # the device sums gradients in FP32: within 1e-3 of the oracle's constants
        ok = np.all(np.abs(g_cs - o_cs) <= 1e-3 * np.maximum(1.0, np.abs(o_cs)), axis=0)
        assert ok.mean() >= 0.9
        return
    same = np.all(g_cs.view(np.uint32) == o_cs.view(np.uint32), axis=0)
    check_paths(same, m, f"full programs cap={cap} n={n}:")
    assert np.array_equal(g_pr[same], p_ref[same])


@pytest.mark.parametrize("n,tapes", [(1, 40), (63, 2049), (65, 100), (128, 4097), (129, 100), (256, 4096), (256, 4097),
                                     (257, 100), (513, 600)])
def test_noalloc_eval_prepares_the_dataset(oracle, gpr, n, tapes):
    """gpr_eval_loglik_noalloc_async where its dataset constants move between the evaluator's
    workgroups and a launch of their own, with equal deviations and one per point, against
    gpr_eval_loglik; the normaliser is the same FP64 sum in another order, of logs that may
    differ by an ulp from the host libm's logf."""
    import torch
    cap = 128
    O, V, L = batch(oracle, cap)
    idx = np.arange(tapes) % O.shape[1]
    O, V, L = O[:, idx].copy(), V[:, idx].copy(), L[idx].copy()
    dO, dV, dL = dev(O), dev(V), dev(L)
    for uneven in (False, True):
        data = dataset(n, uneven)
        ref = torch.zeros(tapes, dtype=torch.float64, device="cuda")
        with gpr.Context(cap=cap) as ctx:
            ctx.set_data([data], [1])
            ctx.eval_loglik_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), tapes, cap, gpr.SCHED_WAVE, ref.data_ptr())
        x, y, sd = (dev(v) for v in data)
        out = torch.full((tapes,), 7.0, dtype=torch.float64, device="cuda")
        say(f"no-alloc dataset n={n} tapes={tapes} uneven={uneven}")
        gpr.eval_loglik_noalloc_async(0, x.data_ptr(), y.data_ptr(), sd.data_ptr(), n, dO.data_ptr(), dV.data_ptr(),
                                      dL.data_ptr(), tapes, cap, gpr.SCHED_WAVE, out.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        ref, out = ref.cpu().numpy(), out.cpu().numpy()
        assert np.all(np.isfinite(ref)) and np.all(np.abs(out - ref) <= 1e-9 * np.maximum(np.abs(ref), n))
    # a deviation that is not positive: every result NaN
    o2 = dev(out)
    bad = dev(np.where(np.arange(n) == n - 1, 0.0, 1.0).astype(np.float32))
    gpr.eval_loglik_noalloc_async(0, x.data_ptr(), y.data_ptr(), bad.data_ptr(), n, dO.data_ptr(), dV.data_ptr(),
                                  dL.data_ptr(), tapes, cap, gpr.SCHED_WAVE, o2.data_ptr(), None)
    torch.cuda.synchronize()
    assert not np.any(np.isfinite(o2.cpu().numpy()))


def pairs_tape(length, shift):
    """x, then two leaves, their operator and an addition, moved a token at a time by the
    negations in front; negations fill the rest."""
    toks = ["X"] + ["NEG"] * shift
    c = ("CONST", 0.5)
    k = 0
    while len(toks) + 4 <= length:
        a, b = [("X", "X"), ("X", c), (c, "X"), (c, c)][k % 4]
        toks += [a, b, ("SUB", "MUL", "ADD")[k % 3], ("ADD", "SUB")[k % 2]]
        k += 1
    return toks + ["NEG"] * (length - len(toks))


@pytest.mark.parametrize("n", [20, 64, 65, 200, 700])
def test_two_leaves_and_their_operator(oracle, gpr, n):
    """Every pair of leaves with every operator, at every offset from the last lane of each half
    tape: exactly rounded operations, 1e-6 of max(|LL|, n) as above."""
    import torch
    cap = 128
    tapes = [pairs_tape(length, s) for length in (4, 61, 62, 63, 64, 65, 66, 126, 127, 128) for s in range(min(length, 13))]
    arrs = [oracle.tape_arrays(t) for t in tapes]
    N = len(arrs)
    O, V = np.zeros((cap, N), dtype=np.uint8), np.zeros((cap, N), dtype=np.float32)
    for i, (o, v) in enumerate(arrs):
        O[:len(o), i], V[:len(v), i] = o, v
    L = np.array([len(o) for o, _ in arrs], dtype=np.int32)
    d = dataset(n, uneven=True)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([d], [1])
        out = torch.zeros(N, dtype=torch.float64, device="cuda")
        say(f"two leaves and an operator n={n} tapes={N}")
        dO, dV, dL = dev(O), dev(V), dev(L)
        ctx.eval_loglik_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), N, cap, gpr.SCHED_WAVE, out.data_ptr())
        got = out.cpu().numpy()
    ref = np.array([oracle.tape_loglik(O[:L[i], i], V[:L[i], i], *d) for i in range(N)])
    assert np.all(np.isfinite(ref))
    assert np.all(np.abs(got - ref) <= 1e-6 * np.maximum(np.abs(ref), n))


@pytest.mark.parametrize("overflow", [False, True])
@pytest.mark.parametrize("n", [7, 64, 130, 300, 700])
def test_exp_log_and_division(oracle, gpr, n, overflow):
    """The handlers of exp, log and division around the magnitude where exp leaves the block, at
    every place of the second half tape's edge: 1e-5 of max(|LL|, n) for the device's exp and
    log; a point where exp overflows makes every LL with it -inf."""
    import torch
    cap = 128
    one, half = ("CONST", 1.0), ("CONST", 0.5)
    bodies = [["X", "EXP", "LOG"], ["X", half, "MUL", "EXP", "X", "X", "MUL", one, "ADD", "DIV", "LOG"],
              ["X", "X", "X", "MUL", one, "ADD", "DIV", "EXP", "X", "ADD"]]
    tapes = [b[:1] + ["NEG"] * pad + b[1:] for b in bodies for pad in (0, 52, 54, 56, 58, 60, 62, 64)]
    arrs = [oracle.tape_arrays(t) for t in tapes]
    N = len(arrs)
    O, V = np.zeros((cap, N), dtype=np.uint8), np.zeros((cap, N), dtype=np.float32)
    for i, (o, v) in enumerate(arrs):
        O[:len(o), i], V[:len(v), i] = o, v
    L = np.array([len(o) for o, _ in arrs], dtype=np.int32)
    x = np.linspace(-20, 20, n).astype(np.float32)
    x[:6] = [87.9, 88.0, 88.3, -87.9, -88.0, -88.3]
    if overflow:
        x[-1] = 89.0
    d = (x, np.zeros(n, dtype=np.float32), np.full(n, 0.5, dtype=np.float32))
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([d], [1])
        out = torch.zeros(N, dtype=torch.float64, device="cuda")
        say(f"exp, log and division n={n} overflow={overflow}")
        dO, dV, dL = dev(O), dev(V), dev(L)
        ctx.eval_loglik_dev(0, dO.data_ptr(), dV.data_ptr(), dL.data_ptr(), N, cap, gpr.SCHED_WAVE, out.data_ptr())
        got = out.cpu().numpy()
    ref = np.array([oracle.tape_loglik(O[:L[i], i], V[:L[i], i], *d) for i in range(N)])
    fin = np.isfinite(ref)
    assert fin.any() and fin.all() == (not overflow) and np.array_equal(fin, np.isfinite(got))
    assert np.all(got[~fin] == -np.inf)
    assert np.all(np.abs(got - ref)[fin] <= 1e-5 * np.maximum(np.abs(ref[fin]), n))
