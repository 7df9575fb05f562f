"""The arrays that a vector step's kernel writes into are checked before their
addresses reach it: dtype, length, shape, contiguity and device of each.  No
GPU is needed: the arrays are DLPack capsules that describe memory on device 0
and own none, and the checks run without an environment."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

from carl_amd import _carl

N_SIM, N_CARS, OBS_DIM = 5, 3, 131
AGENTS = N_SIM * N_CARS
INT, FLOAT, BFLOAT, BOOL = 0, 2, 4, 6    # DLPack type codes
ROCM, CPU = 10, 1                        # DLPack devices


class _Tensor(C.Structure):
    _fields_ = [("data", C.c_void_p), ("device_type", C.c_int32), ("device_id", C.c_int32), ("ndim", C.c_int32),
                ("code", C.c_uint8), ("bits", C.c_uint8), ("lanes", C.c_uint16), ("shape", C.POINTER(C.c_int64)),
                ("strides", C.POINTER(C.c_int64)), ("byte_offset", C.c_uint64), ("manager", C.c_void_p),
                ("deleter", C.c_void_p)]


_kept = []
_new_capsule = C.pythonapi.PyCapsule_New
_new_capsule.restype = C.py_object
_new_capsule.argtypes = [C.c_void_p, C.c_char_p, C.c_void_p]


def described(shape, code, bits, device=ROCM, index=0, strides=None):
    """A capsule describing an array that does not exist."""
    t = _Tensor(0x1000, device, index, len(shape), code, bits, 1, (C.c_int64 * len(shape))(*shape),
                None if strides is None else (C.c_int64 * len(shape))(*strides), 0, None, None)
    _kept.append((t, shape))
    return _new_capsule(C.addressof(t), b"dltensor", None)


ARRAYS = {
    "obs": ((AGENTS, OBS_DIM), FLOAT, 32), "reward": ((AGENTS,), FLOAT, 32), "terminated": ((AGENTS,), BOOL, 8),
    "truncated": ((AGENTS,), BOOL, 8), "done": ((AGENTS,), BOOL, 8), "returns": ((AGENTS,), FLOAT, 32),
    "lengths": ((AGENTS,), INT, 64), "score_difference": ((N_SIM,), INT, 32), "episode_ticks": ((N_SIM,), INT, 32),
    "overtime": ((N_SIM,), BOOL, 8), "step_returns": ((AGENTS,), FLOAT, 32), "step_lengths": ((AGENTS,), INT, 64),
    "step_done": ((AGENTS,), BOOL, 8), "ended": ((4 * (AGENTS + 1),), INT, 32),
}


def check(**changed):
    """_check_vector_outputs on the right arrays, those given replaced."""
    _carl.Env._check_vector_outputs(N_SIM, N_CARS, OBS_DIM,
                                    *(changed[k] if k in changed else described(*v) for k, v in ARRAYS.items()))


def test_the_right_arrays_pass():
    check()
    check(ended=None)
    check(step_returns=None, step_lengths=None, step_done=None)
    shape, code, bits = ARRAYS["obs"]
    check(obs=described(shape, code, bits, strides=(OBS_DIM, 1)))


@pytest.mark.parametrize("name", list(ARRAYS))
def test_every_array_is_checked(name):
    shape, code, bits = ARRAYS[name]
    others = [(FLOAT, 16), (BFLOAT, 16), (FLOAT, 64), (INT, 32), (INT, 8)]
    for other in others:
        if other != (code, bits):
            with pytest.raises(TypeError, match=f"^{name} has an invalid dtype"):
                check(**{name: described(shape, *other)})
    short, spare = (shape[0] - 1, *shape[1:]), (*shape, 1)
    for wrong in (short, spare, ()):
        with pytest.raises(ValueError, match=f"^{name} has an invalid shape"):
            check(**{name: described(wrong, code, bits)})
    with pytest.raises(ValueError, match=f"^{name} must be contiguous"):
        check(**{name: described(shape, code, bits, strides=(2 * shape[-1],) * (len(shape) - 1) + (2,))})
    for device, index in ((CPU, 0), (ROCM, 1)):
        with pytest.raises(ValueError, match=f"^{name} must be on cuda:0"):
            check(**{name: described(shape, code, bits, device, index)})


@pytest.mark.parametrize("name", [k for k in ARRAYS if k != "ended"])
def test_required_arrays_and_groups(name):
    message = "given together" if name.startswith("step_") else "null vector output"
    for absent in (None, 0):
        with pytest.raises(ValueError, match=message):
            check(**{name: absent})


def test_tensors_of_another_default_dtype_are_refused():
    """What torch.empty gives without a dtype, as a program's default has it."""
    before = torch.get_default_dtype()
    try:
        for dtype in (torch.float64, torch.bfloat16, torch.float16):
            torch.set_default_dtype(dtype)
            with pytest.raises(TypeError, match="^obs has an invalid dtype"):
                check(obs=torch.empty(AGENTS, OBS_DIM))
    finally:
        torch.set_default_dtype(before)
    with pytest.raises(ValueError, match="^obs must be on cuda:0"):
        check(obs=torch.empty(AGENTS, OBS_DIM))


def test_the_number_of_arrays():
    with pytest.raises(TypeError, match="14 vector outputs"):
        _carl.Env._check_vector_outputs(N_SIM, N_CARS, OBS_DIM)
