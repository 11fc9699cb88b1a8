"""The kernels' index arithmetic on the CPU, at sizes that a GPU test would take minutes on."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("index") / "libindex.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "index_shim.cpp"), "-o", out])
    L = C.CDLL(out)
    L.shim_point_offset.restype = C.c_uint32
    return L


@pytest.mark.parametrize("kc", [1, 2, 4])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, (1 << 29) + 5, 1 << 30, (1 << 30) + 130, (1 << 31) - 1])
def test_a_chunk_loads_its_own_points(shim, n, kc):
    """Lane l of chunk `base` loads point base + 64 k + l, or the last one: past 2^30 points too,
    where a point's byte offset in the dataset no longer fits 32 bits."""
    chunk = 64 * kc
    last = (n - 1) // chunk * chunk
    for base in sorted({0, last, max(last - chunk, 0), min(last, (1 << 30) // chunk * chunk)}):
        for i in range(chunk):
            at = 4 * base + shim.shim_point_offset(i, n - 1 - base)
            assert at == 4 * min(base + i, n - 1), (n, base, i)


@pytest.mark.parametrize("threads", [64, 128, 256, 512, 1024])
def test_a_launch_holds_fewer_than_2_32_threads(shim, threads):
    groups = shim.shim_max_groups(threads)
    assert groups * threads < 1 << 32 <= (groups + 1) * threads


@pytest.mark.parametrize("groups,threads", [(1, 512), (8388607, 512), (8388608, 512), (1 << 25, 512), (1 << 24, 512),
                                            ((1 << 31) - 1, 64), ((1 << 31) - 1, 512), (16777216, 256)])
def test_launches_cover_every_workgroup_once(shim, groups, threads):
    """The draws (16 threads a chain), MAP copies (8) and per-tape kernels past 2^32 threads."""
    out = (C.c_int * 1024)()
    n = shim.shim_launches(groups, threads, -1, out, 512)
    assert n == -(-groups // (((1 << 32) - 1) // threads))
    at = 0
    for k in range(n):
        assert out[2 * k] == at and out[2 * k + 1] >= 1 and out[2 * k + 1] * threads < 1 << 32
        at += out[2 * k + 1]
    assert at == groups
    if n > 1:
        assert shim.shim_launches(groups, threads, out[2], out, 512) == -5      # an error ends the walk


def test_adjoint_tokens_keep_their_fields(shim):
    """Any byte as op code (what is past the table's 27 stays an unknown one: 35 is no ADD), rows
    to 126, leaf operands to 255."""
    out = (C.c_int * 4)()
    for op in range(256):
        for row, left, right in ((0, 0, 0), (126, 255, 255), (op // 3, 255 - op, op), (127, 128, 254)):
            shim.shim_gtok(op, row, left, right, out)
            assert list(out) == [min(op, 31), row, left, right] and (out[0] == op or op >= 27)
