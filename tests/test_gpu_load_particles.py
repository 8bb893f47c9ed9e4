"""Particles loaded from device arrays: one kernel where it may read them, the
copies otherwise (unaligned arrays, the system's own); same state and step."""
import ctypes as C

import numpy as np
import pytest

from psb_project_amd import scenes
from psb_project_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["aligned", "positions", "unaligned", "own"])
@pytest.mark.parametrize("n", [0, 1, 255, 257, 1000])
def test_load_from_device_arrays(ctx, oracle, n, form):
    from psb_project_amd.system import FluidSystem
    sc = scenes.wcsph_dam_break(n_side=10)
    g, o = FluidSystem(ctx, sc.params, 1000), oracle.OracleSystem(sc.params, 1000)
    x = sc.pos4[:n].copy()
    rng = np.random.default_rng(n)
    v = np.zeros((n, 4), np.float32)
    v[:, :3] = rng.normal(scale=0.3, size=(n, 3))
    h = np.zeros((n, 4), np.float32)
    h[:, :3] = v[:, :3] + rng.normal(scale=0.01, size=(n, 3)).astype(np.float32)
    if form == "positions":
        v[:], h[:] = 0.0, 0.0
    off = 4 if form == "unaligned" else 0
    held = []

    def device(a):
        raw = np.zeros(off + a.nbytes, np.uint8)
        raw[off:] = a.view(np.uint8).ravel()
        d = ctx.array(raw.nbytes)
        if raw.nbytes:
            d.upload(raw)
        held.append(d)
        return C.c_void_p(d.ptr.value + off)

    px, pv, ph = device(x), device(v), device(h)
    if form == "own":
        # state loaded before, then loaded again from the system's own arrays
        g.set_particles(x, v, h)
        a = g.arrays()
        px, pv, ph = (C.c_void_p(q) for q in (a.pos4, a.vel4, a.vel_inter_ap4))
    if form == "positions":
        pv = ph = None
    ctx.sync()
    check(lib().psb_system_set_particles_device(g.handle, n, px, pv, ph))
    s = g.state()
    assert np.array_equal(s["ids"], np.arange(n, dtype=np.uint32))
    for k, ref in (("pos", x), ("vel", v), ("vh", h)):
        assert np.array_equal(s[k], ref), k
    assert not s["density"].any() and not s["pressure"].any()
    if n:
        o.set_particles(x, v, h)
        g.update(2)
        o.update(2)
        gs, os_ = g.state(), o.state()
        for k in ("pos", "vel", "vh", "density", "pressure", "ids"):
            assert np.array_equal(gs[k], os_[k]), k
        assert g.stats()["flags"] == o.stats()["flags"]
