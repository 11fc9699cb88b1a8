"""Reference semantics at the edges of the kernels' chunks and windows, against the oracle:
datasets around 64 points (one chunk; four points per lane on the lane schedule from 65
on), blocks that end inside the five-step cycle of one structure and four constant steps,
and the draws that reject values (the LCG's words are taken 64 at a time)."""
import numpy as np
import pytest

from gpu_util import check_paths, kappa, ll_agree, say


def dataset(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-3, 3, n)
    y = np.sin(x) * 2 + 0.5 * x + rng.normal(0, 0.3, n)
    return x.astype(np.float32), y.astype(np.float32), rng.uniform(0.2, 0.6, n).astype(np.float32)


CASES = [("lane", 1, 1, 5), ("lane", 1, 63, 11), ("lane", 1, 65, 40), ("lane", 0, 64, 13), ("lane", 1, 257, 9),
         ("wave", 0, 1, 1), ("wave", 0, 63, 2), ("wave", 0, 64, 3), ("wave", 0, 65, 4), ("wave", 0, 129, 6),
         ("wave", 0, 257, 9), ("wave", 0, 20, 43)]


@pytest.mark.gpu
@pytest.mark.parametrize("sched,rng,n,steps", CASES)
def test_ref_blocks_match_oracle(oracle, gpr, sched, rng, n, steps):
    x, y, sd = dataset(n, n)
    nch = 67
    hop, hc = oracle.ref_init(3, nch)
    o_hop, o_hc = hop.copy(), hc.copy()
    cfg = oracle.GpoRefCfg(rng, 17)
    m = np.full(nch, np.inf)
    for b in range(3):
        mb = np.zeros(nch)
        p1, l1 = oracle.ref_run_block(cfg, o_hop, o_hc, x, y, sd, b * steps, steps, random_seed=100 + b, margin=mb)
        m = np.minimum(m, mb)
    with gpr.Context(semantics=gpr.SEM_REFERENCE, seed=17, rng=rng,
                     schedule=gpr.SCHED_LANE if sched == "lane" else gpr.SCHED_WAVE) as ctx:
        ctx.set_data([(x, y, sd)], [nch])
        ctx.write_state(hop, hc)
        say(f"ref blocks sched={sched} rng={rng} n={n} steps={steps}")
        for b in range(3):
            ctx.run_block(steps, 100 + b)
        g_hop, g_hc, _, g_pr, g_ll = ctx.read_state()
        st = ctx.stats()
    assert st.steps == 3 * steps * nch and st.struct_proposed == 3 * nch * ((steps + 4) // 5)
    same = np.all(g_hop == o_hop, axis=0) & np.all(g_hc.view(np.uint32) == o_hc.view(np.uint32), axis=0)
    check_paths(same, m, f"{sched} rng={rng} n={n}:")
    c = np.flatnonzero(same)
    assert np.array_equal(g_pr[c], p1[c])
    kap = np.array([kappa(oracle, *oracle.ref_decode(o_hop[:, i].copy(), o_hc[:, i].copy())[:2], x, y, sd) for i in c])
    ok, _ = ll_agree(g_ll[c], l1[c], n, kap, sd)
    assert ok.all()


def test_random_float_product_equals_quotient():
    """random_float is (float)((double)r / 1000000.0) (main.cu:230-232); the kernels take the
    product with 1e-6, which rounds to the same float for every r."""
    r = np.arange(1000000)
    assert np.array_equal((r.astype(np.float32).astype(np.float64) / 1000000.0).astype(np.float32),
                          (r.astype(np.float64) * 1e-6).astype(np.float32))
