"""The stage update from one pair of buffers into another (jfa_rk3_stage_into) and the face-halo fill in
one launch, on the GPU: the update equals, bit for bit, jfa_rk3_stage on copies of the buffers, and the
fill equals the oracle's.  Sizes: one cell more and less than a block of 256 threads, one thread, halos
wider than the grid."""
import numpy as np
import pytest
import torch

from oracle import jxf_oracle as o

pytestmark = pytest.mark.gpu

GRIDS = [((1, 1, 250), 3), ((1, 251, 1), 3), ((257, 1, 1), 3), ((5, 7, 1), 5), ((3, 1, 4), 3), ((2, 3, 1), 3), ((6, 5, 9), 4)]


def _buffers(cells, nh, dtype, seed):
    rng = np.random.default_rng(seed)
    shape = (5,) + tuple(n + 2 * nh if n > 1 else 1 for n in cells)
    W = 1.0 + 0.2 * rng.random(shape)
    U = o.cons_from_prim(W, 1.4)
    return [torch.as_tensor(a, dtype=dtype, device="cuda") for a in (W, U, 1.01 * U, rng.random((5,) + cells))]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("cells, nh", GRIDS)
@pytest.mark.parametrize("stage", [0, 1, 2])
def test_into_equals_in_place(cells, nh, dtype, stage):
    from jaxfluids_amd import _native

    lib, P = _native.load(), _native.ptr
    W, U, Un, rhs = _buffers(cells, nh, dtype, sum(cells) + stage)
    grid = _native.make_grid(cells, nh, (0.1, 0.2, 0.3))
    scheme = _native.make_scheme("PRIMITIVE", "WENO5-JS", "HLLC", "EINFELDT", "ARITHMETIC", _native.dtype_code(W), 1.4,
                                 1e-20)
    W1, U1, W2, U2 = W.clone(), U.clone(), torch.full_like(W, -1.0), torch.full_like(U, -1.0)
    un = P(Un if stage else None)
    assert lib.jfa_rk3_stage(P(U1), un, P(rhs), P(W1), grid, scheme, stage, P(None), 0.01, _native.stream_ptr()) == 0
    assert lib.jfa_rk3_stage_into(P(W), P(U), un, P(rhs), P(W2), P(U2), grid, scheme, stage, P(None), 0.01,
                                  _native.stream_ptr()) == 0
    assert torch.equal(W1, W2) and torch.equal(U1, U2)
    same = (P(W), P(U), un, P(rhs), P(W), P(U2), grid, scheme, stage, P(None), 0.01, _native.stream_ptr())
    assert lib.jfa_rk3_stage_into(*same) == _native.JFA_EINVAL


@pytest.mark.parametrize("types", [("PERIODIC", "PERIODIC"), ("SYMMETRY", "ZEROGRADIENT"), ("ZEROGRADIENT", "SYMMETRY")])
@pytest.mark.parametrize("cells, nh", GRIDS)
def test_halos_match_oracle(cells, nh, types):
    from jaxfluids_amd import _native

    dom = o.Domain(cells, ((0.0, 1.0), (0.0, 1.0), (0.0, 1.0)), nh=nh)
    if any(nh > n for n in cells if n > 1):
        types = ("ZEROGRADIENT", "ZEROGRADIENT")  # the other types need as many cells as halo cells
    s = o.Setup(gamma=1.4, bcs=dict(zip(_native.FACE_LOCATIONS, types * 3)))
    W, U, _, _ = _buffers(cells, nh, torch.float64, sum(cells))
    Wr, Ur = o.halo_update(W.cpu().numpy().copy(), U.cpu().numpy().copy(), dom, s)
    rc = _native.load().jfa_halo_update(_native.ptr(W), _native.ptr(U), _native.make_grid(cells, nh, dom.dx),
                                        _native.bc_array(s.bcs), 1.4, _native.F64, _native.stream_ptr())
    assert rc == 0
    assert np.array_equal(W.cpu().numpy(), Wr)
    assert np.max(np.abs(U.cpu().numpy() - Ur)) <= 4e-16 * np.max(np.abs(Ur))  # cons(W): products and sums of 3 squares
