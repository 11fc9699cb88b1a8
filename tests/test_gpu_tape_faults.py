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
