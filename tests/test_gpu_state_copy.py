"""State copies through the pinned ring: sizes below one piece (2 MB), around one, around the
ring's eight pieces and past several turns of it, in both directions and both semantics."""
import numpy as np
import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu

DATA = (np.linspace(-1, 1, 5).astype(np.float32), np.zeros(5, dtype=np.float32), np.ones(5, dtype=np.float32))


def tapes(gpr, cap, N, seed):
    """Constants joined by additions, of random odd lengths; random values in every row."""
    rng = np.random.default_rng(seed)
    L = (2 * rng.integers(0, (cap + 1) // 2, N) + 1).astype(np.int32)
    t = np.arange(cap)[:, None]
    O = np.where(t == 0, gpr.OP["CONST"], np.where(t % 2 == 1, gpr.OP["X"], gpr.OP["ADD"]))
    O = np.where(t < L[None, :], O, 0).astype(np.uint8)
    return O, rng.normal(size=(cap, N)).astype(np.float32), L


@pytest.mark.parametrize("cap,N", [(32, 1), (32, 1000), (1, 100003), (64, 6398), (64, 6400), (64, 6560), (128, 26000),
                                   (128, 26400), (127, 120001)])
def test_write_and_read_back(gpr, cap, N):
    O, V, L = tapes(gpr, cap, N, N)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([DATA], [N])
        say(f"state copies cap={cap} chains={N}")
        for turn in range(2):
            ctx.write_state(O, V, L)
            o, v, ln, _, _ = ctx.read_state()
            assert np.array_equal(o, O) and np.array_equal(v.view(np.uint32), V.view(np.uint32)) and np.array_equal(ln, L)
            O, V, L = tapes(gpr, cap, N, N + 1)


@pytest.mark.parametrize("N", [1, 7, 20000, 150000])
def test_heaps_write_and_read_back(gpr, N):
    rng = np.random.default_rng(N)
    P = rng.integers(0, 5, (31, N)).astype(np.int32)
    V = rng.normal(size=(31, N)).astype(np.float32)
    with gpr.Context(semantics=gpr.SEM_REFERENCE) as ctx:
        ctx.set_data([DATA], [N])
        say(f"heap state copies chains={N}")
        ctx.write_heap_i32(P, V)
        p, v, _, _ = ctx.read_heap_i32()
    assert np.array_equal(p, P) and np.array_equal(v.view(np.uint32), V.view(np.uint32))


@pytest.mark.parametrize("cap,N", [(32, 50), (64, 90000)])
def test_lowest_bad_chain_is_reported(gpr, cap, N):
    O, V, L = tapes(gpr, cap, N, 3)
    with gpr.Context(cap=cap) as ctx:
        ctx.set_data([DATA], [N])
        ctx.write_state(O, V, L)
        say(f"bad chains cap={cap} chains={N}")
        for bad, text in ((N // 3, "malformed postfix"), (N // 4, "bad op code"), (1, "len out of")):
            if text == "malformed postfix":
                O[0, bad] = gpr.OP["ADD"]
            elif text == "bad op code":
                O[0, bad] = 200
            else:
                L[bad] = 0
            with pytest.raises(Exception, match=f"chain {bad}: {text}"):
                ctx.write_state(O, V, L)
