"""CPU checks of the two-pass PRIMITIVE transpose sweeps (adj_face_kernel, adj_cell_march_kernel,
adj_cell_lane_kernel of jfa_adjoint.h) at the edges of their waves and chunks, through the host build
of the library, against torch autograd of the stage (test_torch_stage, at its tolerance).

A lane wave owns 60 cells of a row with its three halo cells a side (54 cells fill one wave, 55 start
a second, 114 fill two), a marching chunk 8 cells of a column on grids this small (10 cells fill two
chunks, 11 start a third); 3 cells are the fewest that a periodic axis with three halo cells takes.
"""
import pytest

from oracle import jxf_oracle as o
from test_emu_adjoint import FACES, emu  # noqa: F401 - emu: fixture
from test_torch_stage import _compare

PERIODIC = ("PERIODIC",) * 6
WALLS = ("SYMMETRY", "ZEROGRADIENT", "ZEROGRADIENT", "SYMMETRY", "SYMMETRY", "ZEROGRADIENT")


@pytest.mark.parametrize("stencil, riemann", [("WENO5-Z", "HLLC"), ("WENO5-JS", "RUSANOV")])
@pytest.mark.parametrize("cells, bcs", [((54, 1, 1), PERIODIC), ((55, 1, 1), WALLS), ((10, 54, 1), WALLS),
                                        ((11, 55, 1), PERIODIC), ((3, 114, 1), PERIODIC), ((3, 10, 55), WALLS),
                                        ((11, 3, 3), PERIODIC)])
def test_matches_autograd(emu, cells, bcs, stencil, riemann):  # noqa: F811
    dom = o.Domain(cells, ((0.0, 1.0), (0.0, 1.1), (0.0, 0.9)), nh=3)
    s = o.Setup(gamma=1.4, stencil=stencil, variable="PRIMITIVE", riemann=riemann, signal_speed="EINFELDT",
                bcs=dict(zip(FACES, bcs)))
    _compare(emu, dom, s, 1, "march", sum(cells), sum(cells) + 1)
