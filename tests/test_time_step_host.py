"""A step's dt on the host (SimulationManager.do_integration_step): what the manager keeps for it."""
import copy

import pytest
import torch

from oracle import jxf_oracle as o
from test_emu_fused import FACES
from test_gpu_parity import FLUX_CASES, _input_manager, _setup, random_state


def _manager(**kw):
    from jaxfluids_amd import SimulationManager

    s = _setup(FLUX_CASES[0], {f: "PERIODIC" for f in FACES})
    dom, W0 = random_state((9, 8, 7), 3, seed=5, jump=False)
    return SimulationManager(_input_manager(dom, s), **kw), s, dom, W0


def _state(dom, s, W0, dt):
    from jaxfluids_amd.data_types import JaxFluidsBuffers, MaterialFieldBuffers, TimeControlVariables

    W, U = o.create_buffers(W0, dom, s)
    tcv = TimeControlVariables(physical_simulation_time=0.0, simulation_step=0, end_time=1e30, end_step=5,
                               physical_timestep_size=torch.full((1,), dt, dtype=torch.float64, device="cuda"))
    return JaxFluidsBuffers(MaterialFieldBuffers(*(torch.as_tensor(a, device="cuda") for a in (U, W)), None), tcv)


def test_construction_leaves_an_unused_gpu_alone(monkeypatch):
    """A program may build its manager before it chooses a device or forks: where a GPU is there but not in use,
    building one asks for no pinned or device memory and creates no event."""
    def refuse(*args, **kwargs):
        raise AssertionError("the GPU is touched")

    empty = torch.empty
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: False)
    monkeypatch.setattr(torch.cuda, "Event", refuse)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: refuse() if k.get("pin_memory") or k.get("device") else empty(*a, **k))
    _manager()


@pytest.mark.gpu
def test_a_step_within_a_step_keeps_its_own_dt():
    """Two states advanced through one manager, the second while the first one's step is under way: each
    one's time moves by its own dt."""
    sim, s, dom, W0 = _manager(fused=False)
    a, b = _state(dom, s, W0, 1e-3), _state(dom, s, W0, 2e-3)
    sim.do_integration_step(a)  # what the manager keeps from its first step on is there
    kernels, inner = sim._step_kernels, []

    def step_kernels(*args):
        sim._step_kernels = kernels
        inner.append(sim.do_integration_step(b))
        return kernels(*args)

    sim._step_kernels = step_kernels
    dt = float(a.time_control_variables.physical_timestep_size)
    outer = sim.do_integration_step(a)
    assert outer.time_control_variables.physical_simulation_time == dt != 2e-3
    assert inner[0].time_control_variables.physical_simulation_time == 2e-3


@pytest.mark.gpu
def test_copies_of_a_manager_step():
    """copy.deepcopy of a manager that has not stepped yet (its native scheme cannot be copied)."""
    sim, s, dom, W0 = _manager()
    dts = []
    for m in (sim, copy.deepcopy(sim)):
        for _ in range(2):
            out = m.do_integration_step(_state(dom, s, W0, 1e-3))
            assert out.time_control_variables.physical_simulation_time == 1e-3
            dts.append(float(out.time_control_variables.physical_timestep_size))
    assert len(set(dts)) == 1


@pytest.mark.gpu
def test_inference_mode_and_default_device():
    """A manager built or first stepped in inference mode, or with a default device, steps outside of them too."""
    with torch.inference_mode():
        sim, s, dom, W0 = _manager()
        for _ in range(2):
            sim.do_integration_step(_state(dom, s, W0, 1e-3))
    default = torch.get_default_device()
    torch.set_default_device("cuda")
    try:
        other = _manager()[0]
    finally:
        torch.set_default_device(default)
    for m in (sim, other):
        out = m.do_integration_step(_state(dom, s, W0, 1e-3))
        assert out.time_control_variables.physical_simulation_time == 1e-3
