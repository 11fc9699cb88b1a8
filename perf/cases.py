"""The work a user of this package has it do, as timed cases.

Every case goes through the public entry points (gpuropolis_amd.lib.Context and
gpuropolis_amd.autograd) and is a plain dict.  Three kinds of work:

  kind "run"      a sampler run as the command line does it: chains drawn (or loaded from
                  a checkpoint), blocks of MH steps with resampling in between, the state
                  read back.  sampler "walk" and "mala" are the postfix sampler with
                  random-walk and Langevin constant moves, "heap" and "lcg" the
                  reference semantics on Philox streams and on the reference's own LCG.
  kind "eval"     log-likelihoods of a set of tapes on one dataset (entry "context", or
                  "stream": the call that allocates nothing and runs on the caller's stream).
  kind "grad"     log posteriors and their gradients (entry "context", or "torch": the
                  differentiable torch function, forward and backward).

Dataset sizes follow the ones the package is used with: 6 to 250 points for measured
data (the NIST StRD sets among them), up to 1024 for the largest form.
"""
import math

import numpy as np
import torch

from gpuropolis_amd import lib as G
from gpuropolis_amd.autograd import log_posterior

LEAVES = ("X", "CONST", "ONE")
BINARY = ("ADD", "SUB", "MUL", "DIV", "POW", "RSUB", "RDIV", "RPOW")
UNARY = ("NEG", "EXP", "LOG", "INV", "SQRT", "SIN", "ASIN", "COS", "ACOS", "TAN", "ATAN", "ABS", "CADD", "CMUL", "CPOW",
         "CRPOW")
NAMES = ("X", "CONST", "ONE") + BINARY + UNARY
CODE = {n: i for i, n in enumerate(NAMES)}
WITH_CONST = ("CONST", "CADD", "CMUL", "CPOW", "CRPOW")
# the grammar the postfix sampler generates from, and every op a tape may hold
SAMPLER_OPS = (("X", "CONST"), ("ADD", "SUB", "MUL", "DIV", "POW"), ("NEG", "EXP", "LOG"))
ALL_OPS = (LEAVES, BINARY, UNARY)


def listed():
    return [
        # a first look at one small dataset: a thousand chains, short blocks; launches and the
        # length of one chain's serial work decide
        dict(name="run_small", kind="run", sampler="walk", sets=1, lo=32, hi=32, chains=1024, cap=32, blocks=2, steps=100,
             graph=False, resume=False),
        # the usual production run: many chains on one measured dataset
        dict(name="run_large", kind="run", sampler="walk", sets=1, lo=250, hi=250, chains=131072, cap=64, blocks=2, steps=500,
             graph=False, resume=False),
        # a batch of uneven datasets in one context, blocks replayed from a graph
        dict(name="run_batched", kind="run", sampler="walk", sets=48, lo=6, hi=250, chains=2048, cap=128, blocks=2, steps=250,
             graph=True, resume=False),
        # the largest form: long programs, up to 1024 points, Langevin moves
        dict(name="run_langevin", kind="run", sampler="mala", sets=64, lo=16, hi=1024, chains=1024, cap=128, blocks=2,
             steps=200, graph=False, resume=False),
        # the reference's own sampler over a batch of measured datasets, median resampling
        dict(name="run_heap", kind="run", sampler="heap", sets=18, lo=6, hi=236, chains=2048, cap=31, blocks=2, steps=250,
             graph=False, resume=False),
        # the same sampler on the reference's random numbers, at the command line's default N
        dict(name="run_lcg", kind="run", sampler="lcg", sets=1, lo=37, hi=37, chains=1024, cap=31, blocks=1, steps=100,
             graph=False, resume=False),
        # a saved run taken up again: checkpoint to the device, one block, state back
        dict(name="run_resumed", kind="run", sampler="walk", sets=7, lo=50, hi=250, chains=8191, cap=64, blocks=1, steps=200,
             graph=False, resume=True),
        # scoring a handful of programs from a serving loop
        dict(name="eval_few", kind="eval", entry="stream", tapes=48, cap=32, n=32, ops="sampler", uneven=False),
        # scoring an ensemble of samples on the dataset it was drawn for
        dict(name="eval_many", kind="eval", entry="context", tapes=100003, cap=64, n=250, ops="sampler", uneven=False),
        # long programs over every op, a large dataset with a deviation of its own per point
        dict(name="eval_long", kind="eval", entry="context", tapes=6007, cap=128, n=1021, ops="all", uneven=True),
        # gradients of long programs on a large dataset
        dict(name="grad_long", kind="grad", entry="context", tapes=6007, cap=128, n=1021, ops="sampler", uneven=False),
        # constants fitted by a torch optimiser: value and gradient through autograd
        dict(name="grad_torch", kind="grad", entry="torch", tapes=4099, cap=32, n=37, ops="all", uneven=False),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "eval", "eval", "grad", "grad"])
    if kind == "run":
        sampler = rng.choice(["walk", "walk", "mala", "heap", "lcg"])
        top = 1024 if sampler == "mala" else 250
        lo = _between(rng, 6, top)
        hi = _between(rng, lo, top)
        sets = _between(rng, 1, 24)
        steps = rng.randint(20, 300)
        # chain-steps of one pass, so that no drawn run outlasts the largest listed one
        budget = {"walk": 2.0e7, "mala": 4.0e6, "heap": 4.0e6, "lcg": 1.0e5}[sampler]
        blocks = rng.randint(1, 3)
        if sampler == "lcg":            # its blocks are a chain of serial steps over every point
            steps = max(4, min(steps, 3000 // (hi * blocks)))
        chains = _between(rng, 33, max(64, min(65536 // sets, min(16384, int(budget / (sets * steps * blocks))))))
        cap = 31 if sampler in ("heap", "lcg") else rng.choice([16, 32, 47, 64, 100, 128])
        resume = sampler in ("walk", "mala") and rng.random() < 0.25
        graph = sampler != "lcg" and rng.random() < 0.35
        return dict(kind="run", sampler=sampler, sets=sets, lo=lo, hi=hi, chains=chains, cap=cap, blocks=blocks, steps=steps,
                    graph=graph, resume=resume)
    n = _between(rng, 5, 1024)
    cap = rng.choice([8, 16, 32, 47, 64, 100, 128])
    tapes = _between(rng, 1, min(65536, int(6.0e6 / n)))
    entry = rng.choice(["stream", "context"]) if kind == "eval" else rng.choice(["context", "torch"])
    return dict(kind=kind, entry=entry, tapes=tapes, cap=cap, n=n, ops=rng.choice(["sampler", "all"]), uneven=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _dataset(rng, n, uneven=False):
    """A smooth curve with noise; deviations equal, or one per point."""
    x = rng.uniform(-5.0, 5.0, n)
    a, b, c = rng.normal(0.0, 1.0, 3)
    f = 2.0 * np.sin(x + a) + 0.5 * b * x + c
    sd = rng.uniform(0.05, 0.5, n) if uneven else np.full(n, 0.2)
    y = f + sd * rng.normal(0.0, 1.0, n)
    return x.astype(np.float32), y.astype(np.float32), sd.astype(np.float32)


def _structure(rng, want, groups):
    """A random postfix program of `want` tokens over the groups (leaves, binary, unary)."""
    leaves, binary, unary = groups
    toks, need = [], 1
    while need > 0:
        room = want - len(toks) - need       # tokens left beyond the leaves still owed
        u = rng.random()
        if room >= 2 and u < 0.6:
            toks.append(binary[rng.integers(len(binary))])
            need += 1
        elif room >= 1 and u < 0.85:
            toks.append(unary[rng.integers(len(unary))])
        elif need > 1 or room == 0:
            toks.append(leaves[0] if rng.random() < 0.5 else leaves[rng.integers(1, len(leaves))])
            need -= 1
    return toks[::-1]


def _depth(toks):
    d = most = 0
    for t in toks:
        d += 1 if t in LEAVES else (-1 if t in BINARY else 0)
        most = max(most, d)
    return most


def _walk64(toks, cs, x, lib, fit=None):
    """The program's value in the type of its inputs; cs: one value (or [m, 1] column) per
    token.  fit: applied to every token's value."""
    st = []
    for t, c in zip(toks, cs):
        if fit and st:
            st[-1] = fit(st[-1])
        if t == "X":
            st.append(x)
        elif t == "CONST":
            st.append(c + 0.0 * x)
        elif t == "ONE":
            st.append(1.0 + 0.0 * x)
        elif t in BINARY:
            b, a = st.pop(), st.pop()
            st.append({"ADD": lambda: a + b, "SUB": lambda: a - b, "MUL": lambda: a * b, "DIV": lambda: a / b,
                       "POW": lambda: a ** b, "RSUB": lambda: b - a, "RDIV": lambda: b / a, "RPOW": lambda: b ** a}[t]())
        else:
            a = st.pop()
            st.append({"NEG": lambda: -a, "EXP": lambda: lib.exp(a), "LOG": lambda: lib.log(a), "INV": lambda: 1.0 / a,
                       "SQRT": lambda: lib.sqrt(a), "SIN": lambda: lib.sin(a), "ASIN": lambda: lib.arcsin(a),
                       "COS": lambda: lib.cos(a), "ACOS": lambda: lib.arccos(a), "TAN": lambda: lib.tan(a),
                       "ATAN": lambda: lib.arctan(a), "ABS": lambda: abs(a), "CADD": lambda: a + c, "CMUL": lambda: c * a,
                       "CPOW": lambda: a ** c, "CRPOW": lambda: c ** a + 0.0 * a}[t]())
    return st[0]


def _tapes(rng, count, cap, ops, x, valid):
    """An ensemble of `count` tapes: structures shared as after resampling, constants that
    scatter around their structure's.  Programs are finite on the data and of moderate size,
    as a posterior's are; unless `valid`, one structure in ten is not (a proposal outside the
    domain of a log or a power)."""
    groups = SAMPLER_OPS if ops == "sampler" else ALL_OPS
    x64 = np.asarray(x if valid else x[:: max(1, len(x) // 128)], dtype=np.float64)
    x32 = x64.astype(np.float32)
    pool, centre = [], []
    with np.errstate(all="ignore"):
        for k in range(min(192, max(8, count // 4))):
            want = int(round(math.exp(rng.uniform(0.0, math.log(cap)))))
            for _ in range(80):
                toks = _structure(rng, want, groups)
                if _depth(toks) > G.MAX_DEPTH:
                    continue
                c = (rng.standard_normal(len(toks)) * 2.0).astype(np.float32)
                f, g = _walk64(toks, list(c.astype(np.float64)), x64, np), _walk64(toks, list(c), x32, np)
                fine = np.isfinite(f)
                if np.all(fine) and np.all(np.abs(f) < 1e3) and np.all(np.abs(f - g) <= 1e-5 * (1.0 + np.abs(f))):
                    break
                if not valid and k % 10 == 9 and np.isnan(f).mean() > 0.2 and np.array_equal(fine, np.isfinite(g)):
                    break
            else:
                continue
            pool.append(toks)
            centre.append(c)
    which = rng.integers(0, len(pool), count)
    length = np.array([len(p) for p in pool], dtype=np.int32)
    code = np.zeros((cap, len(pool)), dtype=np.uint8)
    mid = np.zeros((cap, len(pool)), dtype=np.float32)
    for i, (p, c) in enumerate(zip(pool, centre)):
        code[:len(p), i] = [CODE[t] for t in p]
        mid[:len(p), i] = [v if t in WITH_CONST else 0.0 for t, v in zip(p, c)]
    cs = mid[:, which] * (1.0 + 0.02 * rng.standard_normal((cap, count), dtype=np.float32))
    cs = cs.astype(np.float32)
    if valid:       # a tape that its scatter took near a pole goes back to its structure's constants
        with np.errstate(all="ignore"):
            for i, p in enumerate(pool):
                mine = np.flatnonzero(which == i)
                f = np.broadcast_to(_walk64(p, [v[:, None] for v in cs[:len(p), mine]], x[None, :], np), (len(mine), len(x)))
                mine = mine[~np.all(np.abs(f) < 1e3, axis=1)]
                cs[:, mine] = mid[:, i:i + 1]
    return code[:, which].copy(), cs, length[which].copy(), pool, which


def _tape_inputs(case, seed):
    rng = np.random.default_rng(seed)
    data = _dataset(rng, case["n"], case["uneven"])
    return (data,) + _tapes(rng, case["tapes"], case["cap"], case["ops"], data[0], case["kind"] == "grad")


def _run_config(case, seed):
    kw = dict(seed=int(seed), cap=case["cap"])
    if case["sampler"] == "mala":
        kw.update(proposal=G.PROP_MALA, eps=0.01)
    if case["sampler"] in ("heap", "lcg"):
        kw = dict(seed=int(seed), semantics=G.SEM_REFERENCE, resample=G.RS_QUANTILE,
                  rng=G.RNG_LCG if case["sampler"] == "lcg" else G.RNG_PHILOX)
    return kw


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "run":
        sizes = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["sets"])).round().astype(int)
        data = [_dataset(rng, n) for n in sizes]
        chains = [case["chains"]] * case["sets"]
        caps = None
        if case["sets"] > 1 and case["sampler"] in ("walk", "mala"):
            caps = [max(1, case["cap"] >> (2 - d % 3)) for d in range(case["sets"])]
        ctx = G.Context(**_run_config(case, seed))
        ctx.set_data(data, chains, caps)
        saved = None
        if case["resume"]:
            parts = [_tapes(rng, k, caps[d] if caps else case["cap"], "sampler", data[d][0], False)[:3] for d, k in enumerate(chains)]
            rows = case["cap"]
            saved = (np.concatenate([np.pad(p[0], ((0, rows - p[0].shape[0]), (0, 0))) for p in parts], axis=1),
                     np.concatenate([np.pad(p[1], ((0, rows - p[1].shape[0]), (0, 0))) for p in parts], axis=1),
                     np.concatenate([p[2] for p in parts]))
        return dict(case=case, ctx=ctx, saved=saved)
    (x, y, sd), ops, cs, length, _, _ = _tape_inputs(case, seed)
    dev = dict(case=case, ops=torch.from_numpy(ops).cuda(), cs=torch.from_numpy(cs).cuda(), length=torch.from_numpy(length).cuda())
    if case["entry"] == "stream":
        dev["data"] = [torch.from_numpy(v).cuda() for v in (x, y, sd)]
        dev["ll"] = torch.empty(case["tapes"], dtype=torch.float64, device="cuda")
        return dev
    dev["ctx"] = G.Context(cap=case["cap"])
    dev["ctx"].set_data([(x, y, sd)], [1])
    if case["entry"] == "context":
        dev["ll"] = torch.empty(case["tapes"], dtype=torch.float64, device="cuda")
        dev["grad"] = torch.empty_like(dev["cs"])
    else:
        dev["cs"].requires_grad_(True)
    torch.cuda.synchronize()
    return dev


# ------------------------------------------------------------------ one pass
def _run_sampler(case, ctx, saved):
    ctx.set_clock(0, 0)
    if saved is None:
        ctx.init_chains()
    else:
        ctx.write_state(*saved)
    if case["graph"]:
        ctx.run_blocks_graph(case["blocks"], case["steps"])
    else:
        for b in range(case["blocks"]):
            ctx.run_block(case["steps"], 12345 + b)
            ctx.resample()
    ops, cs, length, prior, ll = ctx.read_state()
    out = dict(ops=ops, cs=cs, prior=prior, ll=ll)
    if case["sampler"] in ("walk", "mala"):
        out["length"] = length
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "run":
        return _run_sampler(case, state["ctx"], state["saved"])
    ops, cs, length, cap, count = state["ops"], state["cs"], state["length"], case["cap"], case["tapes"]
    if case["kind"] == "eval":
        ll = state["ll"]
        if case["entry"] == "stream":
            x, y, sd = state["data"]
            G.eval_loglik_noalloc_async(0, x.data_ptr(), y.data_ptr(), sd.data_ptr(), case["n"], ops.data_ptr(), cs.data_ptr(),
                                        length.data_ptr(), count, cap, G.SCHED_AUTO, ll.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream)
        else:
            state["ctx"].eval_loglik_dev(0, ops.data_ptr(), cs.data_ptr(), length.data_ptr(), count, cap, G.SCHED_AUTO,
                                         ll.data_ptr())
        return ll
    if case["entry"] == "context":
        state["ctx"].grad_logpost_dev(0, ops.data_ptr(), cs.data_ptr(), length.data_ptr(), count, cap, state["grad"].data_ptr(),
                                      state["ll"].data_ptr())
        return state["ll"], state["grad"]
    lp = log_posterior(state["ctx"], 0, ops, cs, length)
    grad, = torch.autograd.grad(lp.sum(), cs)
    return lp.detach(), grad


def _tape_range(v):
    """Tape values are 32-bit numbers: what is beyond their range is infinite, or zero."""
    v = torch.where(v.abs() > 3.4028235e38, torch.sign(v) * math.inf, v)
    return torch.where(v.abs() < 1e-45, torch.zeros_like(v), v)


def exact(case, seed):
    """Likelihoods and gradients in 64 bits.  A sampler run's result is a random path: its
    programs, and the values that belong to them, have no 64-bit counterpart."""
    if case["kind"] == "run":
        return None
    (x, y, sd), ops, cs, length, pool, which = _tape_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, y, sd = (torch.from_numpy(v).to(dev, torch.float64) for v in (x, y, sd))
    norm = torch.sum(0.5 * math.log(2.0 * math.pi) + torch.log(sd))
    grads = case["kind"] == "grad"
    ll = np.empty(case["tapes"], dtype=np.float64)
    grad = np.zeros(cs.shape, dtype=np.float64)
    for i, toks in enumerate(pool):
        mine = np.flatnonzero(which == i)
        for part in np.array_split(mine, max(1, len(mine) * len(x) * len(toks) // 40_000_000)):
            if not len(part):
                continue
            c = torch.from_numpy(cs[:len(toks), part]).to(dev, torch.float64)
            cols = [v[:, None].requires_grad_(grads) for v in c]
            f = _walk64(toks, cols, x[None, :], torch, _tape_range) + torch.zeros(len(part), 1, dtype=torch.float64, device=dev)
            v = -torch.sum(_tape_range((f - y) ** 2) / (2.0 * sd ** 2), dim=1) - norm
            v = torch.where(torch.isfinite(v), v, -math.inf)
            held = [k for k, t in enumerate(toks) if t in WITH_CONST]
            if grads:
                v = v - len(toks) * math.log(10.0) - math.log(10.0) * sum(t in WITH_CONST[1:] for t in toks)
                for k in held:
                    v = v - math.log(math.pi) - torch.log1p(cols[k][:, 0] ** 2)
                if held:
                    got = torch.autograd.grad(v.sum(), [cols[k] for k in held], allow_unused=True)
                    for k, g in zip(held, got):
                        if g is not None:
                            grad[k, part] = g[:, 0].cpu().numpy()
            ll[part] = v.detach().cpu().numpy()
    return (ll, grad) if grads else ll


def work(case):
    if case["kind"] == "run":
        total = case["sets"] * case["chains"]
        state = total * (5 * case["cap"] + 20)
        # every proposal is judged on at least a wave's worth of points; programs hold about
        # ten tokens, half of them operators, and four more operations make the Gaussian term
        points = min(64, int((case["lo"] * case["hi"]) ** 0.5))
        return dict(bytes=(2 if case["resume"] else 1) * state + 12 * case["sets"] * case["hi"],
                    flops=total * case["blocks"] * case["steps"] * points * (5 + 4) * (2 if case["sampler"] == "mala" else 1))
    tokens = (case["cap"] - 1) / math.log(case["cap"])       # mean of the lengths' law
    out = 8 + (4 * case["cap"] if case["kind"] == "grad" else 0)
    return dict(bytes=case["tapes"] * (5 * tokens + 4 + out) + 12 * case["n"],
                flops=case["tapes"] * case["n"] * (0.5 * tokens + 4) * (2 if case["kind"] == "grad" else 1))
