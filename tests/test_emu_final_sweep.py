"""CPU checks of the FINAL kernel of the fused stage (jfa_fused.h: the last two sweeps and the
finish in one pass) and of the MARCH kernel's packed columns, through the host build of the
library (tests/emu): one RK3 step with the next CFL time step against the oracle's step (FP64,
relative L-inf <= 1e-12), every load and store checked against the registered buffers.

The grids sit at the kernel's edges: rows of one wavefront, one cell more and one less, rows shorter
than the packed wave's step and rows that several waves share, chunks with a remainder, every
orientation of a 2-D domain, the smallest extents that the halos allow.
"""
import dataclasses

import numpy as np
import pytest

from oracle import jxf_oracle as o
from test_emu_fused import FACES, check_step, emu, fused_step  # noqa: F401 - emu: fixture
from test_gpu_parity import random_state, rel

SCHEMES = {
    "z-charprim-hllc": dict(stencil="WENO5-Z", variable="CHAR-PRIMITIVE", riemann="HLLC"),
    "js-charprim-rusanov": dict(stencil="WENO5-JS", variable="CHAR-PRIMITIVE", riemann="RUSANOV"),
    "js-prim-hllc": dict(stencil="WENO5-JS", variable="PRIMITIVE", riemann="HLLC"),
}
BCS = {
    "periodic": {f: "PERIODIC" for f in FACES},
    "mixed": {"east": "ZEROGRADIENT", "west": "SYMMETRY", "north": "SYMMETRY", "south": "ZEROGRADIENT",
              "top": "SYMMETRY", "bottom": "SYMMETRY"},
}
GRIDS = [(4, 5, 64), (3, 4, 65), (4, 3, 63), (5, 6, 11), (3, 3, 3), (6, 1, 13), (1, 7, 58), (9, 66, 1), (11, 128, 1),
         (5, 130, 1)]


@pytest.mark.parametrize("bcs", list(BCS))
@pytest.mark.parametrize("cells", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
@pytest.mark.parametrize("scheme", list(SCHEMES))
def test_step(emu, scheme, cells, bcs):  # noqa: F811
    s = o.Setup(gamma=1.4, signal_speed="EINFELDT", frozen_state="ARITHMETIC", bcs=BCS[bcs], **SCHEMES[scheme])
    dom, W0 = random_state(cells, 3, seed=sum(cells), jump=False)
    check_step(emu, dom, s, W0)


ONE_DIMENSIONAL = [n for N in (17, 64, 100) for n in ((1, N, 1), (1, 1, N))]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("cells", ONE_DIMENSIONAL, ids=["x".join(map(str, g)) for g in ONE_DIMENSIONAL])
@pytest.mark.parametrize("variable", ["PRIMITIVE", "CHAR-PRIMITIVE"])
@pytest.mark.parametrize("riemann, bcs", [("HLLC", "periodic"), ("RUSANOV", "mixed")])
def test_one_dimensional(emu, riemann, bcs, variable, cells, dtype):  # noqa: F811
    """A domain along y or z alone has no second axis to walk along: the step and the right-hand side
    against the oracle, every access inside the registered buffers.  FP32 storage: a step's state is
    rounded to float three times, the right-hand side of the rounded state once."""
    from jaxfluids_amd import _native

    s = o.Setup(gamma=1.4, signal_speed="EINFELDT", frozen_state="ARITHMETIC", stencil="WENO5-Z", variable=variable,
                riemann=riemann, bcs=BCS[bcs])
    dom, W0 = random_state(cells, 3, seed=sum(cells), jump=False)
    if dtype == np.float64:
        check_step(emu, dom, s, W0)
    W, U = o.create_buffers(W0, dom, s)
    dt = o.compute_dt(W, dom, s)
    Wr, _ = o.rk3_step(W, U, dt, dom, s)
    Wg, _, _ = fused_step(emu, dom, s, W, U, dt, dtype=dtype)
    I = dom.interior
    assert rel(Wg[I].astype(np.float64), Wr[I]) < (1e-12 if dtype == np.float64 else 1e-6)

    emu.jfa_compute_rhs.restype, emu.jfa_compute_rhs.argtypes = _native.SIGNATURES["jfa_compute_rhs"]
    emu.jfa_rhs_workspace_bytes.restype, emu.jfa_rhs_workspace_bytes.argtypes = _native.SIGNATURES["jfa_rhs_workspace_bytes"]
    code = _native.F64 if dtype == np.float64 else _native.F32
    grid = _native.make_grid(dom.cells, dom.nh, dom.dx)
    scheme = _native.make_scheme(s.variable, s.stencil, s.riemann, s.signal_speed, s.frozen_state, code, s.gamma,
                                 s.eps_stencil)
    Wd, Ud = np.ascontiguousarray(W.astype(dtype)), np.ascontiguousarray(U.astype(dtype))
    rhs = np.full((5,) + dom.cells, np.nan, dtype=dtype)
    ws = np.zeros(emu.jfa_rhs_workspace_bytes(grid, code), dtype=np.uint8)
    emu.emu_clear_ranges()
    for a in (Wd, Ud, rhs, ws):
        emu.emu_add_range(a.ctypes.data, a.nbytes)
    assert emu.jfa_compute_rhs(Wd.ctypes.data, Ud.ctypes.data, grid, scheme, 0.0, rhs.ctypes.data, ws.ctypes.data,
                               ws.nbytes, None) == 0
    assert emu.emu_violations() == 0, hex(emu.emu_first_violation())
    want = o.compute_rhs(Wd.astype(np.float64), Ud.astype(np.float64), dom, s, 0.0)
    assert rel(rhs.astype(np.float64), want) < (1e-12 if dtype == np.float64 else 1e-6)


def test_common_options_match_the_general_kernels(emu):  # noqa: F811
    """The interpolation limiter sends the same scheme through MARCH + INNER; on a state that it does
    not touch both routes give the same step to rounding."""
    s = o.Setup(gamma=1.4, signal_speed="EINFELDT", frozen_state="ARITHMETIC", bcs=BCS["mixed"], **SCHEMES["z-charprim-hllc"])
    dom, W0 = random_state((5, 6, 20), 4, seed=3, jump=False)
    W, U = o.create_buffers(W0, dom, s)
    dt = o.compute_dt(W, dom, s)
    a = fused_step(emu, dom, s, W, U, dt)
    b = fused_step(emu, dom, dataclasses.replace(s, interpolation_limiter=True), W, U, dt)
    I = dom.interior
    assert np.max(np.abs(a[0][I] - b[0][I])) <= 1e-13 * np.max(np.abs(b[0][I]))
    assert abs(a[2] - b[2]) <= 1e-14 * dt
