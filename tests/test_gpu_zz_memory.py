"""Runs beside a large allocation (needs the GPU): what the state of a run needs is enough for it,
and what a faster kernel keeps beside it is left out when the memory is short.  The test holds most
of the device's memory itself while it runs.
"""
import contextlib
import ctypes

import numpy as np
import pytest

from fdtd3d_amd.config import parse_args
from fdtd3d_amd.engine import Batch, Engine, load_library

pytestmark = pytest.mark.gpu

# TMz with PML, FP64: 0.1 GB a word of every cell; 8 words of state, eps and mu
ARGS = "--2d-tmz --size x:3600,y:3500 --use-pml --pml-size x:10,y:10 --point-source x:1800,y:1700 --point-source-ez " \
       "--time-steps 12"
WORD = 3600 * 3500 * 8


@contextlib.contextmanager
def only(leave):
    """Holds the free device memory but `leave` bytes (64 MB more at most)."""
    lib = load_library()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    held = []
    try:
        for _ in range(40):
            assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            if free.value <= leave + (64 << 20):
                break
            p = ctypes.c_void_p()
            if lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(max(32 << 20, int(0.9 * (free.value - leave))))) == 0:
                held.append(p)
        print(f"[gpu] {free.value / 1e9:.2f} GB left free", flush=True)
        assert free.value <= leave + (64 << 20)
        yield
    finally:
        for p in held:
            lib.hipFree(p)
        lib.hipGetLastError()


def _fields(eps, calls):
    eng = Engine(parse_args(ARGS.split(), precision=8))
    try:
        eng.set_material("eps", eps)
        eng.set_material("mu", eps)
        eng.prepare()
        for n in calls:
            eng.step(n)
        return {c: eng.field_raw(c) for c in ("Ez", "Hx", "Hy", "Dz")}
    finally:
        eng.close()


def test_2d_run_in_short_memory(engine_lib):
    """12 words a cell free: the state and the materials fit (8), the second buffers and factors of
    the register tiles do not (20).  The run goes on, with the fields of the run in ample memory."""
    eps = np.random.default_rng(2).uniform(1.0, 3.0, size=(3600, 3500))
    ref = _fields(eps, [12])
    with only(12 * WORD):
        got = _fields(eps, [12])
    for c, v in ref.items():
        assert np.array_equal(got[c], v), c
    assert np.abs(ref["Ez"]).max() > 0


def test_batch_in_short_memory(engine_lib):
    """17 words a cell free: the batch's two buffers and the materials fit (14), the factors of the
    register tiles do not (6 more).  The batch goes on with its other launches, long enough to tune
    them, with the fields of a single run."""
    eps = np.random.default_rng(2).uniform(1.0, 3.0, size=(3600, 3500))
    ref = _fields(eps, [70])
    with only(17 * WORD):
        b = Batch([parse_args(ARGS.split(), precision=8)])
        try:
            b.set_material(0, "eps", eps)
            b.set_material(0, "mu", eps)
            b.prepare()
            b.step(3)
            b.step(67)
            got = {c: b.field(0, c) for c in ref}
        finally:
            b.close()
    for c, v in ref.items():
        assert np.array_equal(got[c], v), c


def test_factors_for_one_part_of_complex_fields(engine_lib):
    """9 words a cell free at yee_prepare: the imaginary part, prepared first, gets its factors (6) and
    the real part does not.  Both parts then take half steps, step for step."""
    eps = np.random.default_rng(2).uniform(1.0, 3.0, size=(3600, 3500))

    def fields(ctx):
        cfg = parse_args(ARGS.split(), precision=8)
        cfg.complex_fields = True
        eng = Engine(cfg)
        try:
            eng.set_material("eps", eps)
            with ctx:
                eng.prepare()
                eng.step(12)
            return {f"{part} {c}": e.field_raw(c) for part, e in (("real", eng), ("imag", eng.imag())) for c in ("Ez", "Hx", "Dz")}
        finally:
            eng.close()

    ref = fields(contextlib.nullcontext())
    got = fields(only(9 * WORD))
    for c, v in ref.items():
        assert np.array_equal(got[c], v), c
    assert min(np.abs(ref["real Ez"]).max(), np.abs(ref["imag Ez"]).max()) > 0
