"""One call's input tensors are ordered before the engine's stream by the first
of them: which exports carry the stream, and that inputs still being computed
on a side stream arrive whole."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import carl_amd
from carl_amd import workloads

pytestmark = pytest.mark.gpu

N_SIM, CARS = 33, 2


class Producer:
    """Another library's array: orders its own data."""

    def __init__(self, tensor, log):
        self.tensor, self.log = tensor, log

    def __dlpack__(self, stream=None):
        self.log.append(("other", stream))
        return torch.Tensor.__dlpack__(self.tensor, stream=stream)


def given(seed):
    state = workloads.random_reset_state(np.random.default_rng(seed), N_SIM, CARS)
    return {k: torch.from_numpy(v).cuda() for k, v in state.items()}


@pytest.mark.parametrize("foreign", [None, "car_position"])
def test_which_exports_order_the_stream(monkeypatch, foreign):
    env = carl_amd.Env(N_SIM, 1, 1, 0, 8, True, False, False)
    inputs, log = given(1), []
    export = torch.Tensor.__dlpack__

    def logged(self, *args, **kwargs):
        log.append(("torch", kwargs.get("stream")))
        return export(self, *args, **kwargs)

    if foreign:
        inputs[foreign] = Producer(inputs[foreign], log)
    monkeypatch.setattr(torch.Tensor, "__dlpack__", logged)
    env.apply_reset_state(**inputs)
    at = next((i for i, (who, _) in enumerate(log) if who == "other"), None)
    assert (at is not None) == bool(foreign)
    torch_only = [s for who, s in log if who == "torch"]
    engine = env.stream
    if foreign is None:
        assert torch_only == [engine] + [-1] * (len(inputs) - 1)
    else:
        # the first tensor, the other producer (and its tensor), then the tensor after it
        assert log[0] == ("torch", engine) and log[at] == ("other", engine)
        assert log[at + 1:at + 3] == [("torch", engine), ("torch", engine)]
        assert all(s == -1 for _, s in log[1:at] + log[at + 3:])


@pytest.mark.parametrize("masked", [False, True])
def test_inputs_still_being_computed(masked):
    want = carl_amd.Env(N_SIM, 1, 1, 0, 8, True, False, False)
    late = carl_amd.Env(N_SIM, 1, 1, 0, 8, True, False, False)
    inputs = given(2)
    mask = {"reset_mask": torch.arange(N_SIM, device="cuda") % 3 != 1} if masked else {}
    torch.cuda.synchronize()
    want.apply_reset_state(**inputs, **mask)
    want.synchronize()
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        for _ in range(20):
            a = (a @ a) * 1e-3
        zero = (a[0, 0] * 0).nan_to_num()
        args = {k: (v + zero.to(v.dtype)) if v.dtype != torch.bool else v ^ (zero != 0) for k, v in inputs.items()}
        if masked:
            mask = {"reset_mask": mask["reset_mask"] ^ (zero != 0)}
        late.apply_reset_state(**args, **mask)
    late.synchronize()
    assert want.export_state() == late.export_state()
