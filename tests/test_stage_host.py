"""main_amd/csrc/mpcx_stage.hip on the host, with a stand-in for the runtime.

The device blocks the drop-ins keep between calls, with a device heap of a set
size: bounded, the longest unused go first, and given back when anything else
of the library finds no memory.  Copies between host arrays and the device:
the stand-in's streams run them as late as the code may rely on, so a slot
that is used again too soon shows."""
import ctypes as C
import glob
import os
import re

import numpy as np
import pytest

from tests.stage_host import HERE, Stage, rng_bytes

MB = 1 << 20
SLOT, LIMIT = 2 * MB, MB   # a slot; the smallest copy through the ring


@pytest.fixture(scope="module")
def stage(tmp_path_factory):
    return Stage(tmp_path_factory.mktemp("stage"))


def test_blocks_are_reused(stage):
    stage.reset()
    a = stage.get(10 * MB)
    stage.put(a)
    assert stage.get(9 * MB) == a and stage.c.t_mallocs() == 1


def test_another_size_drives_out_the_longest_unused(stage):
    """600 MB of one system's blocks, then calls of another size: kept from the first on."""
    stage.reset()
    old = [stage.get(100 * MB) for _ in range(6)]
    for b in old:
        stage.put(b)
    assert stage.c.t_used() <= 512 * MB
    for _ in range(2):
        new = [stage.get(30 * MB) for _ in range(3)]
        for b in new:
            stage.put(b)
        assert stage.c.t_used() <= 512 * MB
    assert stage.c.t_mallocs() == 9   # the second call's come from the first's
    assert stage.get(100 * MB) in old[2:]   # and the newer ones of the old are still there
    stage.reset()
    big = stage.get(600 * MB)
    stage.put(big)   # more than the cache holds: straight back
    assert stage.c.t_used() == 0


def test_an_allocation_takes_the_cached_memory_back(stage):
    stage.reset(heap=1000 * MB)
    for b in [stage.get(100 * MB) for _ in range(5)]:
        stage.put(b)
    p = stage.c.t_alloc(800 * MB)
    assert p is not None and stage.c.t_used() == 800 * MB
    assert stage.c.t_alloc(300 * MB) is None   # nothing left to give back: an error, as hipMalloc's
    stage.c.t_free(C.c_void_p(p))


def test_every_allocation_goes_through_it():
    for path in glob.glob(os.path.join(HERE, "..", "main_amd", "csrc", "*")):
        if os.path.basename(path) == "mpcx_stage.hip":
            continue
        with open(path) as f:
            code = re.sub(r"//[^\n]*|\"[^\"\n]*\"", "", f.read())
        assert "hipMalloc(" not in code, path


@pytest.mark.parametrize("out", [0, 1])
def test_pinned_arrays_go_straight_over_the_link(stage, out):
    """A pinned array beside a pageable one and a pinned one to be widened."""
    stage.reset()
    sizes = [8 * MB + 24, 5 * MB + 8, 4 * MB]
    dev = [rng_bytes(n, n) for n in sizes]
    host = [np.zeros(n, np.uint8) for n in sizes]
    src, dst = (dev, host) if out else (host, dev)
    for k in range(2):
        src[k][:] = rng_bytes(sizes[k], 3 + k)
    wide = np.zeros(MB, np.int64)
    dev[2] = np.random.default_rng(9).integers(-2**31, 2**31, MB, dtype=np.int64).astype(np.int32)
    host[2] = wide if out else None
    stage.pin(host[0])
    stage.pin(wide)
    assert stage.copy(host, dev, out, widen=[0, 0, out]) == 0
    assert stage.c.t_direct() == sizes[0]
    for k in range(2):
        assert np.array_equal(dst[k], src[k])
    if out:
        assert np.array_equal(wide, dev[2])


def test_the_ring_serves_one_device_after_another(stage):
    stage.reset()
    a, b = rng_bytes(40 * MB + 8, 1), np.zeros(40 * MB + 8, np.uint8)
    for k in range(4):
        stage.c.t_device(k % 2)
        b[:] = 0
        assert stage.copy([b], [a], 1) == 0 and np.array_equal(a, b)
    assert stage.c.t_host_mallocs() == 1 and stage.c.t_events() == 16
    stage.reset()
    assert stage.c.t_events() == 0


@pytest.mark.parametrize("out", [0, 1])
@pytest.mark.parametrize("n", [4096, 9 * MB, 40 * MB])
def test_no_exception_leaves_a_copy(stage, n, out):
    """Each host allocation of a copy fails in turn: the copy is done without it
    or returns an error, and the next one works."""
    a, b = rng_bytes(n, 1), np.zeros(n, np.uint8)
    w = np.zeros(MB, np.int64)
    host = [b, w] if out else [a, None]
    dev = [a if out else b, np.arange(MB, dtype=np.int32)]
    for k in range(64):
        stage.reset()
        b[:] = 0
        rc = stage.copy(host, dev, out, widen=[0, out], fail_at=k)
        if rc < 500:
            assert rc == 0
            break   # no more than k allocations
        assert rc < 1000 or np.array_equal(a, b)
        b[:] = 0
        assert stage.copy(host, dev, out, widen=[0, out]) == 0 and np.array_equal(a, b)
    assert k >= 1 or n < LIMIT   # (a small plain copy allocates nothing)


@pytest.mark.parametrize("out", [0, 1])
@pytest.mark.parametrize("sizes", [[8], [LIMIT - 8], [LIMIT], [SLOT, SLOT + 8], [4 * SLOT - 8, 24, 4 * SLOT + 16], [16 * SLOT],
                                   [16 * SLOT + 8], [7 * MB, 7 * MB, 7 * MB, 7 * MB, 7 * MB, 7 * MB + 8],
                                   [33 * SLOT + 40], [50 * SLOT]])
def test_copies_round_trip(stage, sizes, out):
    """One array and several, up to three times round the ring, into and out of the device."""
    stage.reset()
    src = [rng_bytes(n, n) for n in sizes]
    dst = [np.zeros(n, np.uint8) for n in sizes]
    host, dev = (dst, src) if out else (src, dst)
    assert stage.copy(host, dev, out) == 0
    assert all(np.array_equal(a, b) for a, b in zip(src, dst))
    assert stage.c.t_host_mallocs() == (1 if sum(sizes) >= LIMIT else 0)
