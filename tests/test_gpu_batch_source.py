"""One-launch forms over a hierarchy against their per-patch calls, bit for
bit: the source of every patch (enl_batch_add_source), the microphones
(enl_batch_sample_mics) and the FP32 form's store of patches of every size."""
import ctypes
import math
import time

import numpy as np
import pytest
import torch

from enlightning_amd import _lib, amr
from enlightning_amd import source as SRC
from enlightning_amd.gas import Gas
from enlightning_amd.hierarchy import DeviceHierarchy
from tests import devops as D

pytestmark = pytest.mark.gpu

if D.DRY:
    pytest.skip("the one-launch forms have no CPU stand-in", allow_module_level=True)


def hierarchy(n0=96, tile0=40):
    tags = np.zeros((n0, n0), np.int32)
    tags[20:33, 10:41] = 1
    tags[70:72, 80:95] = 1
    h = amr.build(n0, 4, 4, 1.0, tags, tile0=tile0)
    rng = np.random.default_rng(1)
    d = DeviceHierarchy(h, Gas())
    d.load_initial(None, [rng.uniform(1.0, 2.0, size=(5, p.Ny, p.Nx)) for p in h.patches],
                   [rng.uniform(0.0, 1.0, size=(p.Ny, p.Nx)) for p in h.patches])
    return h, d


@pytest.mark.parametrize("src", [
    SRC.Source(mode=SRC.PULSE, type=SRC.POINT, spread=0.05, pos=(0.3, 0.6)),
    SRC.Source(mode=SRC.DRIVEN, type=SRC.POINT, spread=0.05, pos=(0.3, 0.6)),
    SRC.Source(mode=SRC.PULSE, type=SRC.SINE, spread=0.05, sine_amp=0.1, sine_freq=9.0),
    SRC.Source(mode=SRC.PULSE, type=SRC.LIGHTNING, spread=0.02,
               coords=np.array([[0.1, 0.9, 0.4, 0.5], [0.4, 0.5, 0.35, 0.2], [0.35, 0.2, 0.7, 0.1]])),
    SRC.Source(mode=SRC.PULSE, type=SRC.LIGHTNING, coords=np.zeros((0, 4))),
])
def test_source_of_every_patch_in_one_launch(src):
    h, a = hierarchy()
    _, b = hierarchy()
    a.add_source(src, 5, 2, 1e-4)
    st = src.to_struct()
    D2 = ctypes.c_double * 2
    for p in h.patches:
        base = ctypes.c_void_p()
        _lib.check(b.lib.enl_batch_patch_state(b.handle, p.pid, None, None, None, ctypes.byref(base)))
        dx = h.dx(p.level)
        _lib.check(b.lib.enl_add_source(*p.box, D2(p.box[0] * dx, p.box[2] * dx), D2(dx, dx), ctypes.byref(st), 5, 2,
                                        1e-4, ctypes.c_void_p(base.value + 8 * (p.g + p.g * p.Nx)), p.Nx))
    _lib.check(b.lib.enl_batch_prepare(b.handle, b._reflect()))
    assert all(np.array_equal(x, y) for x, y in zip(a.sources(), b.sources()))
    a.close()
    b.close()


def test_bad_sources_are_refused():
    _, d = hierarchy()
    for bad in (dict(mode=3), dict(type=7), dict(mode=SRC.DRIVEN, type=SRC.SINE)):
        with pytest.raises(RuntimeError):
            d.add_source(SRC.Source(**bad), 0, 0, 1e-4)
    d.close()


def mic_entries(h, d, x, y):
    """(microphone, level, patch, value) in the order of the reference's files:
    per level and patch every microphone within the patch's bounds."""
    out = []
    P = [v[0] for v in d.gather(0x20, ghosted=False)]
    for lev in range(h.nlevels):
        dx = h.dx(lev)
        for p in h.level_patches(lev):
            lo, hi = (p.box[0] * dx, p.box[2] * dx), ((p.box[1] + 1) * dx, (p.box[3] + 1) * dx)
            for k in range(len(x)):
                if lo[0] <= x[k] <= hi[0] and lo[1] <= y[k] <= hi[1]:
                    i, j = min(int((x[k] - lo[0]) / dx), p.nx - 1), min(int((y[k] - lo[1]) / dx), p.ny - 1)
                    out.append((k, lev, p.pid, P[p.pid][j, i]))
    return out


def microphones(h, nm):
    """nm places in and around the domain, some on cell and patch edges; the
    first on the corner that most patches of both levels share."""
    rng = np.random.default_rng(nm)
    x, y = rng.uniform(-0.1, 1.1, size=(2, nm))
    x[::3], y[::5] = np.round(x[::3] * 96) / 96, np.round(y[::5] * 96) / 96
    fine = [(a * h.dx(1), b * h.dx(1)) for p in h.level_patches(1) for a in (p.box[0], p.box[1] + 1)
            for b in (p.box[2], p.box[3] + 1)]
    x[0], y[0] = max(fine, key=lambda c: sum(
        p.box[0] * h.dx(p.level) <= c[0] <= (p.box[1] + 1) * h.dx(p.level)
        and p.box[2] * h.dx(p.level) <= c[1] <= (p.box[3] + 1) * h.dx(p.level) for p in h.patches))
    return x, y


@pytest.mark.parametrize("nm", [1, 127, 400])
def test_microphones_in_one_call(nm):
    h, d = hierarchy()
    x, y = microphones(h, nm)
    want = [[] for _ in range(nm)]
    for k, lev, pid, v in mic_entries(h, d, x, y):
        want[k].append((lev, pid, v))
    assert len(want[0]) > 2 and {lev for lev, _, _ in want[0]} == {0, 1}
    assert d.sample_mics(x, y) == want
    d.close()


@pytest.mark.parametrize("room", [0, 1, 129])
def test_microphones_beyond_the_callers_room(room):
    """The count of all entries comes back whatever the room, with the first
    `room` of them and nothing behind; the wrapper calls again with more."""
    h, d = hierarchy()
    x, y = microphones(h, 400)
    want = mic_entries(h, d, x, y)
    assert len(want) > 129
    mic, level, pid = (np.full(room + 2, -7, np.int32) for _ in range(3))
    val = np.full(room + 2, -7.0)
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
    n = d.lib.enl_batch_sample_mics(d.handle, 400, ptr(x), ptr(y), room, ptr(mic), ptr(level), ptr(pid), ptr(val))
    assert n == len(want)
    assert list(zip(mic[:room], level[:room], pid[:room], val[:room])) == want[:room]
    assert all((a[room:] == -7).all() for a in (mic, level, pid, val))
    d.close()
    # the wrapper starts with room for two entries per microphone and level: a
    # corner on which four patches of each level meet has eight
    quarters = [(0, 11, 0, 11), (12, 23, 0, 11), (0, 11, 12, 23), (12, 23, 12, 23)]
    fine = [(32, 47, 32, 47), (48, 63, 32, 47), (32, 47, 48, 63), (48, 63, 48, 63)]
    h = amr.from_boxes(24, 4, 4, 1.0, [(0, *q) for q in quarters] + [(1, *q) for q in fine])
    d = DeviceHierarchy(h, Gas())
    d.load_initial(None, [np.full((5, p.Ny, p.Nx), 1.1 + p.pid) for p in h.patches])
    got = d.sample_mics([0.5], [0.5])[0]
    assert len(got) == 8 and [(0, *q) for q in got] == mic_entries(h, d, [0.5], [0.5])
    d.close()


@pytest.mark.parametrize("origin", [(0.0, 0.0), (2.5, 0.75), (-3.0, -0.25), (-0.5, 8.0)])
def test_microphones_on_a_domain_of_any_origin(origin):
    """A batch made through the C ABI with its lower corner at `origin`: the
    entries are those of enl_sample_mics called patch by patch with the same
    geometry.  dx is a power of two, so every bound is exact."""
    h, whole = hierarchy(64, 24)
    lib, desc = whole.lib, np.zeros(len(h.patches), dtype=_lib.PATCH_DESC_DTYPE)
    for p in h.patches:
        dx = h.dx(p.level)
        desc[p.pid] = (p.level, p.box, (origin[0] + p.box[0] * dx, origin[1] + p.box[2] * dx), (dx, dx))
    handle = ctypes.c_void_p()
    _lib.check(lib.enl_batch_create(len(desc), desc.ctypes.data_as(ctypes.POINTER(_lib.EnlPatchDesc)), h.g, h.ratio,
                                    ctypes.byref(handle)))
    rng = np.random.default_rng(5)
    nm = 90
    x, y = origin[0] + rng.uniform(-0.3, 1.3, nm), origin[1] + rng.uniform(-0.3, 1.3, nm)
    x[::4] = origin[0] + np.round((x[::4] - origin[0]) * 64) / 64  # on cell and patch edges
    want, P = [], []
    for p in h.patches:
        P.append(rng.uniform(1.0, 2.0, size=(p.Ny, p.Nx)))
        a = ctypes.c_void_p(P[-1].ctypes.data)
        _lib.check(lib.enl_batch_copy_state(handle, p.pid, 1, None, a, None, None))
    for lev in range(h.nlevels):
        dx = h.dx(lev)
        for p in h.level_patches(lev):
            lo = desc[p.pid]["xlo"]
            hi = (lo[0] + p.nx * dx, lo[1] + p.ny * dx)
            g = p.g
            v, hit = SRC.sample_mics(p.box, lo, hi, (dx, dx), x, y,
                                     torch.from_numpy(np.ascontiguousarray(P[p.pid][g:-g, g:-g])).cuda())
            torch.cuda.synchronize()
            v, hit = v.cpu().numpy(), hit.cpu().numpy()
            want += [(k, lev, p.pid, v[k]) for k in np.nonzero(hit)[0]]
    assert len({m for m, *_ in want}) > nm // 4 and max(m[1] for m in want) == 1
    room = len(want) + 50
    mic, level, pid = (np.full(room, -1, np.int32) for _ in range(3))
    val = np.zeros(room)
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
    n = lib.enl_batch_sample_mics(handle, nm, ptr(x), ptr(y), room, ptr(mic), ptr(level), ptr(pid), ptr(val))
    got = [(mic[k], level[k], pid[k], val[k]) for k in range(n)]
    _lib.check(lib.enl_batch_destroy(handle))
    whole.close()
    assert got == want


@pytest.mark.parametrize("n0,tile0", [(96, 40), (200, 200), (72, 24)])  # (24 + 8)^2: whole chunks of 256
def test_fp32_load_and_store_of_every_patch(n0, tile0):
    """Load carries the FP64 perturbation of the interior, store adds the
    ambient back: amb + (w - amb) on the interior, amb + float(w - amb) in the
    ghosts and for p and T."""
    h, d = hierarchy(n0, tile0)
    gas = d.gas
    rows = lambda lev: (-4, np.linspace(1.1, 1.3, h.ncells(lev) + 8), np.linspace(-1, 1, h.ncells(lev) + 8),
                        np.linspace(300, 360, h.ncells(lev) + 8))
    d.set_ambient(rows)
    d.fp32_prepare()
    before = d.gather(0x7F)
    # p and T of the ambient, update_state.m4:88-105 as the library's host forms them (c_lr = 0)
    ambient_p = lambda r, rs: gas.c * gas.c * ((r - gas.rho0) + (gas.gamma1 - 1) / (2 * gas.rho0) * (
        (r - gas.rho0) * (r - gas.rho0)) + r / gas.c_p * (rs / r)) + gas.p0
    ambient_T = lambda r, rs: gas.T0 * math.exp((rs / r - gas.R * math.log(gas.rho0 / r)) / gas.c_v)
    d.fp32_load()
    d.fp32_store()
    after = d.gather(0x7F)
    for p, u, v in zip(h.patches, before, after):
        _, r, rs, rt = rows(p.level)
        at = slice(p.box[2], p.box[3] + 2 * p.g + 1)
        g = p.g
        rp, rT = (np.array([f(*q) for q in zip(r.tolist(), rs.tolist())]) for f in (ambient_p, ambient_T))
        for k, amb in ((0, r), (1, 0 * r), (2, 0 * r), (3, rs), (4, rt), (5, rp), (6, rT)):
            A = amb[at][:, None]
            pert = u[k] - A
            want = A + pert.astype(np.float32).astype(np.float64)
            if k < 5:
                want[g:-g, g:-g] = (A + pert)[g:-g, g:-g]
            assert np.array_equal(v[k], want), (p.pid, k)
    d.close()


def host_time(f, reps=10):
    """Seconds of one of `reps` calls of f in a row, the best of five rows."""
    f()
    torch.cuda.synchronize()
    best = np.inf
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(reps):
            f()
        torch.cuda.synchronize()
        best = min(best, (time.perf_counter() - t) / reps)
    return best


def test_fp32_load_and_store_fill_the_chip_whatever_the_patches():
    """2048^2 cells in one patch and in 1024 of 64^2: the ghosts of the small
    ones are a quarter more to move, so the one patch takes no longer than
    they do; twice their time is allowed.  (With workgroups counted per patch,
    64 at most, it took seven times as long.)"""
    took = {}
    for tile0 in (64, 2048):
        h = amr.build(2048, 4, 4, 1.0, None, tile0=tile0)
        d = DeviceHierarchy(h, Gas())
        rows = np.ones(2048 + 8)
        d.set_ambient(lambda lev: (-4, 1.2 * rows, 0.1 * rows, 350.0 * rows))
        d.fp32_prepare()
        took[len(h.patches)] = host_time(d.fp32_load) + host_time(d.fp32_store)
        d.close()
    assert took[1] <= 2 * took[1024], took


def test_source_fills_the_chip_whatever_the_patches():
    """A lightning channel of 48 segments, bound by the exponentials of each
    cell, over the same cells: 1.75 times the small patches' time is allowed
    to the one patch.  (With at most 256 workgroups of one wave per SIMD each,
    it took 2.5 times as long.)"""
    seg = np.array([[0.1, 0.9, 0.4, 0.5], [0.4, 0.5, 0.35, 0.2], [0.35, 0.2, 0.7, 0.1]] * 16)
    src = SRC.Source(mode=SRC.PULSE, type=SRC.LIGHTNING, spread=0.02, coords=seg)
    took = {}
    for tile0 in (64, 2048):
        h = amr.build(2048, 4, 4, 1.0, None, tile0=tile0)
        d = DeviceHierarchy(h, Gas())
        took[len(h.patches)] = host_time(lambda: d.add_source(src, 0, 0, 1e-4))
        d.close()
    assert took[1] <= 1.75 * took[1024], took
