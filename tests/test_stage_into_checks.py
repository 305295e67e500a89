"""What jfa_rk3_stage_into and RungeKutta3.perform_stage_integration(primitives=...) refuse, on the CPU: outputs
that overlap an input or one another (the kernel reads and writes through pointers that must not alias), and
primitives that are not laid out as the conservatives are."""
import numpy as np
import pytest
import torch

from test_emu_fused import emu  # noqa: F401 - fixture

CELLS, NH = (4, 3, 5), 3
SHAPE = (5,) + tuple(n + 2 * NH for n in CELLS)


def _call(emu, stage=1, dtype=np.float64, **pointers):
    from jaxfluids_amd import _native

    fn = emu.jfa_rk3_stage_into
    fn.restype, fn.argtypes = _native.SIGNATURES["jfa_rk3_stage_into"]
    size = int(np.prod(SHAPE))
    bufs = {k: np.ones(2 * size, dtype=dtype) for k in ("W", "U", "U_n", "rhs", "W_out", "U_out")}
    emu.emu_clear_ranges()
    for a in bufs.values():
        emu.emu_add_range(a.ctypes.data, a.nbytes)
    at = {k: bufs[k].ctypes.data for k in bufs}
    for k, (other, items) in pointers.items():
        at[k] = at[other] + items * bufs[other].itemsize
    scheme = _native.make_scheme("PRIMITIVE", "WENO5-JS", "HLLC", "EINFELDT", "ARITHMETIC",
                                 _native.F64 if dtype == np.float64 else _native.F32, 1.4, 1e-30)
    return fn(*at.values(), _native.make_grid(CELLS, NH, (0.1, 0.1, 0.1)), scheme, stage, None, 0.01, None)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_overlaps_are_refused(emu, dtype):  # noqa: F811
    from jaxfluids_amd import _native

    size, nrhs = int(np.prod(SHAPE)), 5 * int(np.prod(CELLS))
    for out, other in [("W_out", "W"), ("W_out", "U"), ("U_out", "W"), ("U_out", "U"), ("U_out", "U_n"), ("W_out", "U_n"),
                       ("U_out", "W_out"), ("W_out", "rhs"), ("U_out", "rhs")]:
        n = nrhs if other == "rhs" else size
        for items in (0, 1, n - 1):
            assert _call(emu, dtype=dtype, **{out: (other, items)}) == _native.JFA_EINVAL, (out, other, items)
        assert _call(emu, dtype=dtype, **{out: (other, n)}) == _native.JFA_OK, (out, other)
    assert _call(emu, stage=0, dtype=dtype) == _native.JFA_OK


def test_primitives_must_be_laid_out_as_the_conservatives():
    from jaxfluids_amd.data_types import EulerIntegrationBuffers, IntegrationBuffers
    from jaxfluids_amd.domain import DomainInformation
    from jaxfluids_amd.time_integration import RungeKutta3

    rk = RungeKutta3(nh=NH, inactive_axes=[])
    U = torch.ones(SHAPE, dtype=torch.float64)
    wrap = lambda t: IntegrationBuffers(EulerIntegrationBuffers(t))  # noqa: E731
    rhs = wrap(torch.zeros((5,) + CELLS, dtype=torch.float64))
    dom = DomainInformation.__new__(DomainInformation)
    for W in (U.float(), U[:, 1:], torch.ones(SHAPE[::-1], dtype=torch.float64).permute(3, 2, 1, 0)):
        with pytest.raises(ValueError, match="primitives"):
            rk.perform_stage_integration(wrap(U), rhs, wrap(U), 0.01, 0, None, dom, 1.4, primitives=W)
        with pytest.raises(ValueError, match="primitives"):
            rk.perform_stage_integration(wrap(U), rhs, wrap(U), 0.01, 0, None, dom, 1.4, primitives_out=W, primitives=U)
