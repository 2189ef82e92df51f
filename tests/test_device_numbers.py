"""Numbers that the host hands a step without a wait (ops/slots.py)."""
import pytest
import torch

from jax_llama_amd.ops.slots import device_numbers


def test_on_the_cpu():
    for values in ([3], [1, -2, 70000], (5, 6), range(4)):
        got = device_numbers(values, torch.int32, "cpu")
        assert got.dtype == torch.int32 and got.tolist() == list(values)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 700])
def test_copies_in_flight_keep_their_own_memory(n):
    """Many pending copies behind a stream that is busy: pinned memory is not handed out again before its copy is done."""
    a = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        a = a @ a * 1e-3
    got = [device_numbers(list(range(i, i + n)), torch.long, "cuda") for i in range(200)]
    assert all(t.tolist() == list(range(i, i + n)) for i, t in enumerate(got))
