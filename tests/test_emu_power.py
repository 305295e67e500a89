"""power (jfa_dissipative.h), the x^p of the transport laws, on the CPU: its error against extended
precision and its values outside 0 < x < infinity against pow, and the CFL time step of states with a
negative temperature (CPU emulation of the kernels, tests/emu) against the oracle's NaN.

The error bound is half an ulp of the final rounding and 0.1 ulp for the terms that the series' two-double
sums drop; extended precision adds a thousandth of that."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import jxf_oracle as o
from test_emu_fused import FACES, emu  # noqa: F401 - emu: fixture
from test_gpu_parity import random_state

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
EXPONENTS = (0.5, 0.7, 0.76, 1.5, -0.7, 3.0, -2.0, 2.0, -1.0, 1.0 / 3.0)


@pytest.fixture(scope="module")
def power(tmp_path_factory):
    """power as a vectorised function, built for the host like the emulation."""
    d = tmp_path_factory.mktemp("power")
    src = d / "power.cpp"
    src.write_text('#include "jfa_dissipative.h"\n'
                   "namespace jfa { thread_local char g_last_error[256]; }\n"
                   'extern "C" void power_n(const double* x, double p, double* out, long n, int sgn) {\n'
                   "    for (long i = 0; i < n; ++i)\n"
                   "        out[i] = sgn ? jfa::power<false, true>(x[i], p) : jfa::power<true, false>(x[i], p);\n"
                   "}\n")
    lib = d / "power.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-pthread",
                    "-Wno-unknown-pragmas", "-Wno-attributes", f"-I{os.path.join(HERE, 'emu')}",
                    f"-I{os.path.join(ROOT, 'jaxfluids_amd', 'csrc')}", f"-I{os.path.join(ROOT, 'include')}", str(src),
                    os.path.join(HERE, "emu", "emu_runtime.cpp"), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).power_n
    fn.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_void_p, ctypes.c_long, ctypes.c_int]
    fn.restype = None

    def call(x, p, signed=True):
        x = np.ascontiguousarray(x, dtype=np.float64)
        out = np.empty_like(x)
        fn(x.ctypes.data, p, out.ctypes.data, x.size, int(signed))
        return out

    return call


@pytest.mark.parametrize("signed", [True, False])
@pytest.mark.parametrize("p", EXPONENTS)
def test_error(power, p, signed):
    rng = np.random.default_rng(5)
    x = np.concatenate([np.exp(rng.uniform(-300.0, 300.0, 20000) / max(1.0, abs(p))), rng.uniform(0.5, 2.0, 20000),
                        1.0 + rng.uniform(-1e-7, 1e-7, 4000), [1.0, 0.5, 2.0, np.sqrt(0.5), np.sqrt(2.0)]])
    want = np.power(x.astype(np.longdouble), np.longdouble(p))
    ulp = np.spacing(np.abs(want).astype(np.float64))
    assert np.max(np.abs(power(x, p, signed) - want) / ulp) < 0.6


@pytest.mark.parametrize("p", EXPONENTS)
def test_special_values(power, p):
    x = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -1.0, -0.37, -1e300, -1e-300, -2.5])
    with np.errstate(all="ignore"):
        want = np.power(x, p)
    got = power(x, p)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    number = ~np.isnan(want)
    assert np.array_equal(np.signbit(got[number]), np.signbit(want[number]))
    positive = ~np.signbit(x)  # the faces' variant: from 0 up, and NaN
    assert np.array_equal(power(x[positive], p, False), got[positive], equal_nan=True)
    finite = np.isfinite(want) & (want != 0.0)
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True)
    assert np.all(np.abs(got[finite] - want[finite]) <= 2.0 * np.spacing(np.abs(want[finite])))  # pow itself: 1 ulp


LAWS = {
    "power": o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_exp=0.76, bulk_viscosity=1e-2, prandtl=0.71),
    "power-heat-law": o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_exp=-0.7, kappa_ref=1e-2, kappa_exp=0.5),
    "sutherland": o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_sutherland=0.4, prandtl=0.71),
    # a diffusivity that is a number at any temperature: the wave speed alone is NaN
    "constant": o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_exp=0.0, prandtl=0.71),
    "square": o.Transport(R=1.0, mu_ref=2e-2, T_ref=1.0, mu_exp=2.0, prandtl=0.71),
}


def _transport(tr):
    import dataclasses

    from jaxfluids_amd import _native

    return _native.make_transport(**dataclasses.asdict(tr))


def _negative_pressure_dt(emu, tr):
    """jfa_compute_dt of a state with one cell of negative pressure, and the oracle's."""
    from jaxfluids_amd import _native

    dom, W0 = random_state((8, 8, 8), 3, seed=2, jump=False)
    s = o.Setup(gamma=1.4, bcs={f: "PERIODIC" for f in FACES}, cfl=0.5, transport=tr)
    W, _ = o.create_buffers(W0, dom, s)
    W = np.ascontiguousarray(W)
    W[4, dom.nh + 3, dom.nh + 4, dom.nh + 2] = -0.5
    fn = emu.jfa_compute_dt
    fn.restype, fn.argtypes = _native.SIGNATURES["jfa_compute_dt"]
    dt, ws = np.zeros(1), np.zeros(32, dtype=np.uint8)
    emu.emu_clear_ranges()
    for a in (W, dt, ws):
        emu.emu_add_range(a.ctypes.data, a.nbytes)
    assert fn(W.ctypes.data, _native.make_grid(dom.cells, dom.nh, dom.dx), 1.4, 0.5, o.EPS64, _native.F64, _transport(tr),
              dt.ctypes.data, ws.ctypes.data, None) == 0
    assert emu.emu_violations() == 0
    with np.errstate(all="ignore"):
        return float(dt[0]), float(o.compute_dt(W, dom, s))


def _stage_dt(emu, tr):
    """The next time step of one fused stage so long that it leaves cells of negative pressure."""
    from jaxfluids_amd import _native

    dom, W0 = random_state((8, 8, 8), 3, seed=2, jump=False)
    s = o.Setup(gamma=1.4, stencil="WENO5-Z", variable="PRIMITIVE", riemann="HLLC", signal_speed="EINFELDT",
                bcs={f: "PERIODIC" for f in FACES}, cfl=0.5, transport=tr)
    W, U = (np.ascontiguousarray(a) for a in o.create_buffers(W0, dom, s))
    grid = _native.make_grid(dom.cells, dom.nh, dom.dx)
    scheme = _native.make_scheme(s.variable, s.stencil, s.riemann, s.signal_speed, s.frozen_state, _native.F64, s.gamma,
                                 s.eps_stencil, _transport(tr))
    ws = np.zeros(emu.jfa_stage_workspace_bytes(grid, scheme), dtype=np.uint8)
    Wo, Uo, dt = np.full_like(W, np.nan), np.full_like(U, np.nan), np.zeros(1)
    emu.emu_clear_ranges()
    for a in (W, U, Wo, Uo, ws, dt):
        emu.emu_add_range(a.ctypes.data, a.nbytes)
    P = lambda a: a.ctypes.data  # noqa: E731
    assert emu.jfa_rk3_stage_fused(P(W), P(U), None, P(Wo), P(Uo), grid, scheme, _native.bc_array(s.bcs), 0, None, 0.5,
                                   0.5, o.EPS64, P(dt), P(ws), ws.nbytes, None) == 0
    assert emu.emu_violations() == 0
    Wi = Wo[dom.interior]
    assert np.all(np.isfinite(Wi)) and np.any((Wi[4] < 0.0) & (Wi[0] > 0.0))
    return float(dt[0])


@pytest.mark.parametrize("law", list(LAWS))
def test_negative_temperature_gives_nan_dt(emu, law):  # noqa: F811
    got, want = _negative_pressure_dt(emu, LAWS[law])
    assert np.isnan(want) and np.isnan(got)
    assert np.isnan(_stage_dt(emu, LAWS[law]))
