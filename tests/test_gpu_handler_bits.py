"""The interpreter's handlers of exp, log and division give the bits of the compiler's expf, logf and
division: the rejected and the accepted form of a proposal, the adjoint, the forward-mode pass and the
lane schedule use one or the other.  Compared through the two schedules of the evaluator."""
import numpy as np
import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu


def float_bits(v):
    """Tensor of 32-bit patterns (int64) as floats."""
    import torch
    return torch.where(v >= 1 << 31, v - (1 << 32), v).to(torch.int32).view(torch.float32)


def tapes(gpr, op):
    """Tapes c op k1 * k2 * (or a b / k1 * k2 *) on operands of every kind of bit pattern (signs,
    denormals, infinities and NaN among them): k1 and k2 are powers of two that bring the result to
    [0.5, 4), which is exact, so that the squares of neighbouring results differ."""
    import torch
    bits = torch.arange(0, 1 << 32, 1021, dtype=torch.int64, device="cuda")
    a, b = float_bits(bits), float_bits((bits * 2654435761 + 12345) & 0xffffffff)
    r = {"EXP": a.double().exp(), "LOG": a.double().log(), "DIV": a.double() / b.double()}[op]
    e = torch.log2(r.abs())
    e = torch.where(torch.isfinite(e), e, torch.zeros_like(e)).clamp(-149, 128).floor()
    half = torch.floor(-e / 2)
    one = torch.ones_like(e)
    k1, k2 = (torch.ldexp(one, v).float() for v in (half, -e - half))
    ops = [gpr.OP["CONST"]] * (2 if op == "DIV" else 1) + [gpr.OP[op]] + [gpr.OP["CONST"], gpr.OP["MUL"]] * 2
    cs = torch.zeros((len(ops), len(a)), dtype=torch.float32, device="cuda")
    cs[0] = a
    if op == "DIV":
        cs[1] = b
    cs[-4], cs[-2] = k1, k2
    codes = torch.tensor(ops, dtype=torch.uint8, device="cuda")[:, None].repeat(1, len(a))
    return codes, cs, torch.full((len(a),), len(ops), dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("op", ["EXP", "LOG", "DIV"])
def test_handlers_give_the_bits_of_the_compilers_functions(gpr, op):
    """One point of a dataset, in the first, second, third or fourth register of its lane, carries
    all the weight (the others' rounds to 0 in FP32), so equal likelihoods are equal bits."""
    import torch
    codes, cs, length = tapes(gpr, op)
    cap, N = codes.shape
    sets = [(1, 0), (100, 0), (100, 64), (250, 0), (250, 64), (250, 128), (250, 192)]
    data = []
    for n, point in sets:
        sd = np.full(n, 3e38, dtype=np.float32)
        sd[point] = 0.5
        data.append((np.zeros(n, dtype=np.float32), np.zeros(n, dtype=np.float32), sd))
    wave, lane = (torch.zeros(N, dtype=torch.float64, device="cuda") for _ in range(2))
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data(data, [1] * len(sets))
        torch.cuda.synchronize()
        for d, (n, point) in enumerate(sets):
            say(f"{op} n={n} point {point}: {N} tapes")
            for schedule, out in ((gpr.SCHED_WAVE, wave), (gpr.SCHED_LANE, lane)):
                ctx.eval_loglik_dev(d, codes.data_ptr(), cs.data_ptr(), length.data_ptr(), N, cap, schedule, out.data_ptr())
            assert float(torch.isfinite(lane).double().mean()) > 0.4     # half the logarithms are of negative numbers
            assert bool((wave == lane).all()), (n, point, int((wave != lane).sum()))
