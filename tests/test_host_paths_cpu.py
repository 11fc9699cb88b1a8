"""The library's host code on the CPU, with a stub runtime whose calls can be made to fail: what a
call that falls back on another path leaves behind for the calls after it."""
import ctypes as C
import os
import re
import subprocess
import threading

import numpy as np
import pytest

from gpuropolis_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """The library as a ctypes object: gpr_api.hip's host side over hip_stub.cpp."""
    from gpuropolis_amd import lib as G
    d = str(tmp_path_factory.mktemp("host"))
    flags = [f for f in B.HIP_FLAGS if f != "-O3"] + ["-O1", "--cuda-host-only"]
    objs = []
    for src, extra in ((os.path.join(B.CSRC, "gpr_api.hip"), []), (os.path.join(HERE, "hip_stub.cpp"), ["-x", "hip"])):
        objs.append(os.path.join(d, os.path.basename(src) + ".o"))
        subprocess.check_call([B.HIPCC, *flags, *extra, "-c", src, "-o", objs[-1]], stderr=subprocess.DEVNULL)
    names = subprocess.run(["nm", "--undefined-only", *objs], capture_output=True, text=True, check=True).stdout
    fat = os.path.join(d, "fat.cpp")
    with open(fat, "w") as f:         # the device code that is not there
        for n in sorted(set(re.findall(r"__hip_fatbin_\w+", names))):
            f.write(f'extern "C" char {n}[64] = {{0}};\n')
    so = os.path.join(d, "libhost.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", *objs, fat, "-o", so, "-lpthread"])
    path, loaded = G.LIB_PATH, G._lib
    G.LIB_PATH, G._lib = so, None
    try:
        L = G.load()
        L.stub_fail.argtypes = [C.c_char_p, C.c_int]
        yield G, L
    finally:
        G.LIB_PATH, G._lib = path, loaded


@pytest.mark.parametrize("fails", ["hipEventCreateWithFlags", "hipHostMalloc", ""])
@pytest.mark.parametrize("chains", [64, 20000])
def test_state_copies_without_the_pinned_buffer(host, chains, fails):
    """A state goes the plain way when there is no pinned memory, or no event for its ring, and no
    later call fails for it: a launch reports the runtime's pending error as its own."""
    G, L = host
    cap, n = 64, 40
    x = np.linspace(-1, 1, n).astype(np.float32)
    ops = np.zeros((cap, chains), dtype=np.uint8)
    cs = np.arange(cap * chains, dtype=np.float32).reshape(cap, chains)
    ln = np.ones(chains, dtype=np.int32)
    with G.Context(cap=cap) as ctx:
        ctx.set_data([(x, x, np.ones(n, np.float32))], [chains])
        L.stub_fail(fails.encode(), 1 << 30)
        try:
            ctx.write_state(ops, cs, ln)
            ctx.run_block(5)
            got = ctx.read_state()
            ctx.resample()
        finally:
            L.stub_fail(b"", 0)
        assert np.array_equal(got[0], ops) and np.array_equal(got[1], cs) and np.array_equal(got[2], ln)
        again = ctx.read_state()                  # with what failed before
        assert np.array_equal(again[1], cs) and np.array_equal(again[2], ln)


def test_checked_gradients_side_by_side(host):
    """Each call gets the faults of its own tapes, where threads share a context for all that (the
    fault word is the context's)."""
    G, L = host
    got = {}
    one = np.zeros(8, dtype=np.float64)
    p = one.ctypes.data
    with G.Context(cap=1) as ctx:
        ctx.set_data([(np.ones(1, np.float32),) * 3], [1])

        def calls(want):
            length = np.full(1, want, dtype=np.int32)
            got[want] = [ctx.grad_logpost_checked_dev(0, p, p, length.ctypes.data, 1, 1, p, p) for _ in range(50)]

        threads = [threading.Thread(target=calls, args=(w,)) for w in (0, G.TAPE_OP, G.TAPE_POSTFIX)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert all(set(v) == {want} for want, v in got.items()) and len(got) == 3
