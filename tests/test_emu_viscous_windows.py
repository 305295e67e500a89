"""Viscous sweeps of CONSERVATIVE reconstruction on a periodic domain, on the CPU (tests/emu): the convective
windows are of U, and the dissipative faces wrap onto the interior, so no value of W's halo cells is read
-- here they are NaN -- and the right-hand side is the oracle's of the filled buffer."""
import dataclasses

import numpy as np
import pytest

from oracle import jxf_oracle as o
from test_emu_fused import FACES, TOL, emu  # noqa: F401 - emu: fixture
from test_gpu_parity import random_state, rel


@pytest.mark.parametrize("cells", [(9, 8, 7), (13, 11, 1), (1, 9, 11), (17, 1, 1), (1, 1, 70)])
@pytest.mark.parametrize("stencil", ["WENO5-Z", "TENO5"])
def test_primitive_halos_are_not_read(emu, stencil, cells):  # noqa: F811
    from jaxfluids_amd import _native

    dom, W0 = random_state(cells, 3, seed=5, jump=False)
    tr = o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_exp=0.76, bulk_viscosity=1e-2, prandtl=0.71)
    s = o.Setup(gamma=1.4, bcs={f: "PERIODIC" for f in FACES}, transport=tr, stencil=stencil, variable="CONSERVATIVE",
                riemann="HLLC", signal_speed="EINFELDT", frozen_state="ARITHMETIC")
    W, U = (np.ascontiguousarray(a) for a in o.create_buffers(W0, dom, s))
    want = o.compute_rhs(W, U, dom, s, 0.0)
    assert np.all(np.isfinite(want))
    halo = np.ones(dom.shape, dtype=bool)
    halo[dom.interior[1:]] = False
    W[:, halo] = np.nan
    grid_ = _native.make_grid(dom.cells, dom.nh, dom.dx)
    scheme = _native.make_scheme(s.variable, s.stencil, s.riemann, s.signal_speed, s.frozen_state, _native.F64, s.gamma,
                                 s.eps_stencil, _native.make_transport(**dataclasses.asdict(tr)))
    for name in ("jfa_compute_rhs", "jfa_rhs_workspace_bytes"):
        fn = getattr(emu, name)
        fn.restype, fn.argtypes = _native.SIGNATURES[name]
    rhs = np.full((5,) + dom.cells, np.nan)
    ws = np.zeros(emu.jfa_rhs_workspace_bytes(grid_, _native.F64), dtype=np.uint8)
    emu.emu_clear_ranges()
    for a in (W, U, rhs, ws):
        emu.emu_add_range(a.ctypes.data, a.nbytes)
    assert emu.jfa_compute_rhs(W.ctypes.data, U.ctypes.data, grid_, scheme, 0.0, rhs.ctypes.data, ws.ctypes.data,
                               ws.nbytes, None) == 0
    assert emu.emu_violations() == 0, hex(emu.emu_first_violation())
    assert rel(rhs, want) < TOL
