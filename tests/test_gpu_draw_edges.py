"""Draws and resampling at the sizes where their kernels split the chains: workgroups of 32 and
64 chains, the keys that the median select keeps in registers (4096 chains), row groups of
the copies, and heap draws whose integers are rejected."""
import numpy as np
import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu

X = np.linspace(-1, 1, 6).astype(np.float32)
DATA = (X, (2 * X).astype(np.float32), np.full(6, 0.5, dtype=np.float32))


def bits(a):
    return a.view(np.uint32)


@pytest.mark.parametrize("cap,sizes", [(1, [1]), (7, [63, 1]), (32, [64, 65]), (33, [200, 1, 5, 3, 127]), (128, [300, 129])])
def test_init_and_map_resample(oracle, gpr, cap, sizes):
    with gpr.Context(cap=cap, seed=29, resample_nats=1.0) as ctx:
        ctx.set_data([DATA] * len(sizes), sizes)
        say(f"init and MAP resample cap={cap} chains={sizes}")
        ctx.init_chains()
        i_ops, i_cs, i_ln, _, _ = ctx.read_state()
        ctx.run_block(7)
        g = ctx.read_state()
        ctx.resample()
        r = ctx.read_state()
    c0 = moved = 0
    for n in sizes:
        sl = slice(c0, c0 + n)
        o_ops, o_cs, o_ln = oracle.cfg_init(oracle.make_cfg(cap=cap, seed=29), n, chain0=c0)
        assert np.array_equal(i_ln[sl], o_ln) and np.array_equal(i_ops[:, sl], o_ops)
        assert np.array_equal(bits(i_cs[:, sl].copy()), bits(o_cs))
        h = [a[..., sl].copy() for a in g]
        src = np.zeros(n, dtype=np.int32)
        moved += oracle.lib().gpo_cfg_resample(n, c0, 1, 29, cap, 1.0, oracle.u8(h[0]), oracle.f32(h[1]), oracle.i32(h[2]),
                                               oracle.f64(h[3]), oracle.f64(h[4]), oracle.i32(src))
        for a, b in zip(r, h):
            assert np.array_equal(a[..., sl], b, equal_nan=a.dtype.kind == "f")
        c0 += n
    assert moved > 0 or sum(sizes) < 10


@pytest.mark.parametrize("sizes", [[1, 2], [31, 33], [32, 1023, 1024, 1025], [4095, 4097], [4096, 9001]])
def test_heap_init_and_median_resample(oracle, gpr, sizes):
    with gpr.Context(semantics=gpr.SEM_REFERENCE, seed=31, resample=gpr.RS_QUANTILE) as ctx:
        ctx.set_data([DATA] * len(sizes), sizes)
        say(f"heap init and median resample chains={sizes}")
        ctx.init_chains()
        i_hop, i_hc, _, _, _ = ctx.read_state()
        ctx.run_block(6, 1)
        hop, hc, _, pr, ll = ctx.read_state()
        ctx.resample()
        r_hop, r_hc, _, _, _ = ctx.read_state()
    c0 = 0
    for n in sizes:
        sl = slice(c0, c0 + n)
        o_hop, o_hc = oracle.ref_init(31, n, chain0=c0)
        assert np.array_equal(i_hop[:, sl], o_hop) and np.array_equal(bits(i_hc[:, sl].copy()), bits(o_hc))
        o_hop, o_hc = hop[:, sl].copy(), hc[:, sl].copy()
        p, q, cutoff = pr[sl].copy(), ll[sl].copy(), np.zeros(1)
        oracle.lib().gpo_ref_resample(31, 1, n, c0, oracle.u8(o_hop), oracle.f32(o_hc), oracle.f64(p), oracle.f64(q),
                                      oracle.f64(cutoff), 0)
        assert np.array_equal(r_hop[:, sl], o_hop) and np.array_equal(bits(r_hc[:, sl].copy()), bits(o_hc))
        c0 += n


# (seed, chain) whose initial draw rejects an op (words 1 and 26 of the stream) or an order
# (words 49 and 79), found by search on the CPU: some 3e-7 of chains
@pytest.mark.parametrize("seed,chain", [(3325, 59), (4001, 243), (7735, 273), (6120, 730)])
def test_rejected_heap_draws(oracle, gpr, seed, chain):
    n = chain + 2
    hop, hc = oracle.ref_init(seed, n)
    with gpr.Context(semantics=gpr.SEM_REFERENCE, seed=seed) as ctx:
        ctx.set_data([DATA], [n])
        say(f"rejected draw seed={seed} chain={chain}")
        ctx.init_chains()
        g_hop, g_hc, _, _, _ = ctx.read_state()
    assert np.array_equal(g_hop, hop) and np.array_equal(bits(g_hc), bits(hc))
