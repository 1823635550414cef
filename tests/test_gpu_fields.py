"""Upload (swsph_set_particles) and read-back (swsph_get_fields): every field
in one call against one call per field and against what was uploaded, for
one particle, an odd number (unaligned parts of the staging buffer), and
more than a million (sweeps and copies overlap on two streams); mixed and
uniform time bins (the second key sort is left out), and arrays left out
(defaults)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _parts(n, mixed, seed):
    rng = np.random.default_rng(seed)
    f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)
    return dict(x=rng.uniform(0, 1, (n, 3)), v=rng.normal(size=(n, 3)).astype(
                    np.float32),
                m=f(1, 2), u=f(1, 2), h=f(0.01, 0.05), rho=f(1, 2),
                pressure=f(1, 2), soundspeed=f(1, 2), f=f(-1, 1),
                balsara=f(0, 1), alpha_visc=f(0, 1), alpha_diff=f(0, 1),
                div_v_prev=f(-1, 1),
                time_bin=(rng.integers(1, 30, n) if mixed
                          else np.full(n, 4)).astype(np.int8))


def _get_all(eng, n):
    from swift_amd import FIELDS, lib
    names = list(FIELDS)
    outs = [np.empty((n, 3) if FIELDS[k][2] == 3 else (n,), FIELDS[k][1])
            for k in names]
    ids = (C.c_int * len(names))(*[FIELDS[k][0] for k in names])
    ptr = (C.c_void_p * len(names))(*[o.ctypes.data for o in outs])
    assert lib().swsph_get_fields(eng._h, len(names), ids, ptr) == 0
    return dict(zip(names, outs))


@pytest.mark.parametrize("n,mixed", [(1, False), (999, True), (999, False),
                                     ((1 << 20) + 77, True),
                                     ((1 << 20) + 77, False)])
def test_upload_and_read_back(n, mixed):
    from swift_amd import Engine, HydroProps
    p = _parts(n, mixed, seed=n)
    with Engine(HydroProps(ncell=(5, 5, 5))) as eng:
        eng.set_particles(_parts(max(1, n // 2), not mixed, seed=1))  # old data
        eng.set_particles(p)
        got = _get_all(eng, n)
        for k, v in got.items():
            assert np.array_equal(v, eng.get(k)), k
    up = dict(p, v_full=p["v"], u_full=p["u"])
    for k, v in got.items():
        if k in up:
            assert np.array_equal(v, up[k]), k
        else:
            assert not v.any(), k


def test_optional_arrays_and_errors():
    from swift_amd import Engine, HydroProps, lib
    from swift_amd.engine import _HostParts
    p = _parts(999, True, seed=5)
    hp = _HostParts()
    hp.n = 999
    for k in ("x", "v", "m", "u", "h", "time_bin"):
        setattr(hp, k, p[k].ctypes.data)
    with Engine(HydroProps(ncell=(5, 5, 5))) as eng:
        assert lib().swsph_set_particles(eng._h, C.byref(hp)) == 0
        eng.n = 999
        got = _get_all(eng, 999)
        out = np.empty(999, np.float32)
        ids = (C.c_int * 2)(0, 999)
        ptr = (C.c_void_p * 2)(out.ctypes.data, out.ctypes.data)
        assert lib().swsph_get_fields(eng._h, 2, ids, ptr) == 1
    assert np.array_equal(got["x"], p["x"])
    assert np.all(got["alpha_visc"] == np.float32(0.1))
    for k in ("rho", "pressure", "soundspeed", "f", "balsara", "alpha_diff",
              "div_v_prev"):
        assert not got[k].any(), k


@pytest.mark.parametrize("n", [1, 7, 999, 32767, 32768, 70001])
def test_positions_outside_the_box(n):
    """Refused with the index of the first one, on the host and on the device
    (from 32768 particles on), and the last particles stay."""
    from swift_amd import Engine, HydroProps
    from swift_amd._lib import SwsphError
    good = _parts(n, True, seed=n)
    with Engine(HydroProps(ncell=(5, 4, 3), dim=(1.0, 1.5, 2.0))) as eng:
        eng.set_particles(good)
        for i, k, v in ((0, 0, 1.0), (n // 2, 1, 1.5), (n - 1, 2, 2.0),
                        (n - 1, 0, -1e-300), (n // 3, 2, np.nan),
                        (n // 2, 1, np.inf)):
            bad = _parts(n, True, seed=n)
            bad["x"][i, k] = v
            with pytest.raises(SwsphError, match=f"particle {i} lies outside"):
                eng.set_particles(bad)
            assert np.array_equal(eng.get("x"), good["x"])
        edge = _parts(n, True, seed=n)
        edge["x"][n // 2] = [-0.0, np.nextafter(1.5, 0), np.nextafter(2.0, 0)]
        eng.set_particles(edge)
        assert np.array_equal(eng.get("x"), edge["x"])


@pytest.mark.parametrize("n,names", [
    (1, ("time_bin",)), (262144, ("h", "rho")), (262145, ("h", "rho")),
    (65536, ("h", "x", "h")), (9001, ("time_bin", "x", "rho")),
    (5003, None), (70001, None)])
def test_read_back_sizes(n, names):
    """Fields of uploaded particles in one call, to both sides of the 2 MiB
    that leave the device in one copy, and with the staging buffer filled
    several times; a field may be asked for twice."""
    from swift_amd import FIELDS, Engine, HydroProps, lib
    p = _parts(n, True, seed=n)
    with Engine(HydroProps(ncell=(5, 5, 5))) as eng:
        eng.set_particles(p)
        names = names or [k for k in FIELDS if k in p]
        outs = [np.full((n, 3) if FIELDS[k][2] == 3 else (n,), -1,
                        FIELDS[k][1]) for k in names]
        ids = (C.c_int * len(names))(*[FIELDS[k][0] for k in names])
        ptr = (C.c_void_p * len(names))(*[o.ctypes.data for o in outs])
        for _ in range(2):
            assert lib().swsph_get_fields(eng._h, len(names), ids, ptr) == 0
            for k, o in zip(names, outs):
                assert np.array_equal(o, p[k]), k
                o[...] = -1


def test_small_boxes_hold_little_memory():
    """The staging buffer of a small box follows its size: the buffers of 729
    particles (0.5 MB) take less than 2 MiB in each of 16 engines, with every
    field read back (an engine's stream is the runtime's); fields asked for
    more often than the buffer holds arrive as well."""
    from swift_amd import FIELDS, Engine, HydroProps, lib
    p = _parts(729, True, seed=3)

    def free():  # of the HIP runtime that the library is linked with
        got, total = C.c_size_t(), C.c_size_t()
        assert lib().hipMemGetInfo(C.byref(got), C.byref(total)) == 0
        return got.value

    engines = [Engine(HydroProps(ncell=(3, 3, 3))) for _ in range(16)]
    try:
        before = free()
        for eng in engines:
            eng.set_particles(p)
            for k, v in _get_all(eng, 729).items():
                assert k not in p or np.array_equal(v, p[k]), k
        assert before - free() < 16 * (2 << 20)
        names = 5 * [k for k in FIELDS if k in p]
        outs = [np.full((729, 3) if FIELDS[k][2] == 3 else (729,), -1,
                        FIELDS[k][1]) for k in names]
        ids = (C.c_int * len(names))(*[FIELDS[k][0] for k in names])
        ptr = (C.c_void_p * len(names))(*[o.ctypes.data for o in outs])
        assert lib().swsph_get_fields(engines[0]._h, len(names), ids, ptr) == 0
        for k, o in zip(names, outs):
            assert np.array_equal(o, p[k]), k
    finally:
        for eng in engines:
            eng.close()


@pytest.mark.parametrize("n,names", [
    (1, ("h",)), (70001, ("h",)), (20479, ("x", "rho")), (20481, ("x", "rho")),
    (9001, ("h", "rho", "x")), (70001, ("h", "time_bin", "rho", "u")),
    (87000, ("x",)), (5003, None)])
@pytest.mark.parametrize("where", ["locked", "device", "mixed"])
def test_read_back_to_locked_memory(n, names, where):
    """Outputs in page-locked memory (copied to by the device, or through the
    engine's block where that is shorter), in device memory, and one of them
    pageable among page-locked ones."""
    from swift_amd import FIELDS, Engine, HydroProps, lib
    p = _parts(n, True, seed=n)
    names = names or [k for k in FIELDS if k in p]
    size = [n * FIELDS[k][2] * np.dtype(FIELDS[k][1]).itemsize for k in names]
    at = np.cumsum([0] + [(s + 255) // 256 * 256 for s in size])
    L, buf = lib(), C.c_void_p()
    total = C.c_size_t(int(at[-1]))
    alloc = ((lambda b: L.hipMalloc(b, total)) if where == "device"
             else (lambda b: L.hipHostMalloc(b, total, 0)))
    assert alloc(C.byref(buf)) == 0
    host = np.empty(int(at[-1]), np.uint8)
    try:
        with Engine(HydroProps(ncell=(5, 5, 5))) as eng:
            eng.set_particles(p)
            ptrs = [buf.value + int(o) for o in at[:-1]]
            if where == "mixed":
                ptrs[0] = host.ctypes.data
            ids = (C.c_int * len(names))(*[FIELDS[k][0] for k in names])
            outs = (C.c_void_p * len(names))(*ptrs)
            assert L.swsph_get_fields(eng._h, len(names), ids, outs) == 0
            for k, q, s in zip(names, ptrs, size):
                got = np.empty(p[k].shape, p[k].dtype)
                assert L.hipMemcpy(got.ctypes.data_as(C.c_void_p),
                                   C.c_void_p(q), C.c_size_t(s), 4) == 0
                assert np.array_equal(got, p[k]), k
    finally:
        (L.hipFree if where == "device" else L.hipHostFree)(buf)
