"""Gradient calls on tapes that are not sound programs."""
import threading

import numpy as np
import pytest

from gpu_util import dev, say
from test_gpu_interpreter import dataset

pytestmark = pytest.mark.gpu


def sound_tapes(gpr, cap, n):
    x, c, add, mul = (gpr.OP[k] for k in ("X", "CONST", "ADD", "MUL"))
    ops = np.zeros((cap, n), dtype=np.uint8)
    ops[:5] = np.array([c, x, mul, c, add], dtype=np.uint8)[:, None]
    return ops, np.full((cap, n), 0.5, dtype=np.float32), np.full(n, 5, dtype=np.int32)


@pytest.mark.skip(reason="a context belongs to one host thread (include/gpuropolis.h): a process that had run this aborted "
                         "in the HIP runtime when it destroyed a later context, from a cause not shown")
def test_faults_of_calls_side_by_side(gpr):
    """Threads that share a context: each call gets the faults of its own tapes."""
    import torch
    cap, n, rounds = 32, 512, 400
    ops, cs, ln = sound_tapes(gpr, cap, n)
    bad = ln.copy()
    bad[n // 2] = 4                               # two values left
    got = {}
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(70, False)], [1])
        dops, dcs = dev(ops), dev(cs)

        def calls(name, length):
            grad = torch.empty((cap, n), dtype=torch.float32, device="cuda")
            lp = torch.empty(n, dtype=torch.float64, device="cuda")
            dln = dev(length)
            got[name] = [ctx.grad_logpost_checked_dev(0, dops.data_ptr(), dcs.data_ptr(), dln.data_ptr(), n, cap,
                                                      grad.data_ptr(), lp.data_ptr()) for _ in range(rounds)]

        say("checked gradient calls from four threads")
        threads = [threading.Thread(target=calls, args=(k, bad if k % 2 else ln)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for k in range(4):
        want = gpr.TAPE_POSTFIX if k % 2 else 0
        assert got[k] == [want] * rounds, (k, sum(f != want for f in got[k]))


@pytest.mark.parametrize("cap,n", [(64, 70), (128, 600)])
def test_op_codes_that_are_no_ops(gpr, cap, n):
    """The unchecked gradient of a tape with an unknown op code, anywhere in the byte's range: the
    value is no number, so the posterior is -inf, and the tapes beside it keep their results."""
    import torch
    codes = [len(gpr.OPS), 31] + [32 + k for k in range(32)] + [64, 96, 128, 200, 255]
    x, c, add = (gpr.OP[k] for k in ("X", "CONST", "ADD"))
    N = 5 * len(codes)
    ops, cs, ln = sound_tapes(gpr, cap, N)
    clean = ops.copy()
    where = []
    for k, op in enumerate(codes):
        for at, tape in ((5 * k + 1, [x, op]), (5 * k + 2, [c, x, op, add]), (5 * k + 3, [c] + [op] * (cap - 1))):
            ops[:, at] = 0
            ops[:len(tape), at] = tape
            ln[at] = len(tape)
            where.append(at)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(n, True)], [1])
        dcs = dev(cs)
        say(f"unknown op codes, cap {cap}, n {n}")

        def call(o, length):
            grad = torch.empty((cap, N), dtype=torch.float32, device="cuda")
            lp = torch.empty(N, dtype=torch.float64, device="cuda")
            do, dl = dev(o), dev(length)
            ctx.grad_logpost_dev(0, do.data_ptr(), dcs.data_ptr(), dl.data_ptr(), N, cap, grad.data_ptr(), lp.data_ptr())
            return grad.cpu().numpy(), lp.cpu().numpy()

        want_g, want = call(clean, np.full(N, 5, dtype=np.int32))
        got_g, got = call(ops, ln)
    assert np.all(got[where] == -np.inf)
    rest = np.setdiff1d(np.arange(N), where)
    assert np.array_equal(got[rest], want[rest]) and np.array_equal(got_g[:, rest], want_g[:, rest])


@pytest.mark.parametrize("cap,n", [(16, 1), (64, 70), (128, 600), (128, 1025)])
def test_tapes_that_leave_several_values(gpr, cap, n):
    """The unchecked gradient of tapes that end with 2 to 16 values: no program, so the posterior
    is -inf and the gradient the prior's, and the tapes beside them keep their results."""
    import torch
    x, c, add, neg = (gpr.OP[k] for k in ("X", "CONST", "ADD", "NEG"))
    wrong = [[c] * k for k in range(2, 17)] + [[x, x, x, neg, add] + [c] * 6, [c, x, add, c], [c] * 8 + [add] * 6]
    wrong += [[c] * 16 + [neg] * (cap - 16)] if cap > 16 else []
    N = 3 * len(wrong)
    ops, cs, ln = sound_tapes(gpr, cap, N)
    clean = ops.copy()
    where = np.arange(len(wrong)) * 3 + 1
    for at, tape in zip(where, wrong):
        ops[:, at] = 0
        ops[:len(tape), at] = tape
        ln[at] = len(tape)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([dataset(n, True)], [1])
        dcs = dev(cs)
        say(f"several values left, cap {cap}, n {n}")

        def call(o, length):
            grad = torch.empty((cap, N), dtype=torch.float32, device="cuda")
            lp = torch.empty(N, dtype=torch.float64, device="cuda")
            do, dl = dev(o), dev(length)
            ctx.grad_logpost_dev(0, do.data_ptr(), dcs.data_ptr(), dl.data_ptr(), N, cap, grad.data_ptr(), lp.data_ptr())
            return grad.cpu().numpy(), lp.cpu().numpy()

        want_g, want = call(clean, np.full(N, 5, dtype=np.int32))
        got_g, got = call(ops, ln)
    assert np.all(got[where] == -np.inf)
    for at, tape in zip(where, wrong):       # -2 c / (1 + c^2) at c = 0.5, on the constants only
        want_col = np.zeros(cap, dtype=np.float32)
        want_col[:len(tape)] = np.where(np.array(tape) == c, np.float32(-0.8), np.float32(0))
        assert np.array_equal(got_g[:, at], want_col)
    rest = np.setdiff1d(np.arange(N), where)
    assert np.array_equal(got[rest], want[rest]) and np.array_equal(got_g[:, rest], want_g[:, rest])
