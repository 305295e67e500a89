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
from test_gpu_parity import random_state

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
