"""Cache slots that the host knows."""
from __future__ import annotations

import torch


class HostSlot(int):
    """A cache slot known on the host, with its device copy (``on_device``, int32[1]) made once for all ops of a step: a copy
    per op from pageable host memory waits for everything the stream still has to do, twice per layer."""

    def __new__(cls, value: int, device):
        slot = super().__new__(cls, value)
        slot.on_device = torch.full((1,), int(value), dtype=torch.int32, device=device)
        return slot


def step_slot(slot, device):
    """What a model's step hands to its ops for ``slot`` (an int, or a device tensor, which is returned as it is)."""
    if torch.is_tensor(slot) or isinstance(slot, HostSlot) or torch.device(device).type == "cpu":
        return slot
    return HostSlot(int(slot), device)


def slot_tensor(slot, device) -> torch.Tensor:
    """``slot`` as a device int32[1]."""
    if torch.is_tensor(slot):
        return slot
    if isinstance(slot, HostSlot) and slot.on_device.device == torch.device(device):
        return slot.on_device
    return torch.full((1,), int(slot), dtype=torch.int32, device=device)


def device_numbers(values, dtype, device) -> torch.Tensor:
    """The numbers ``values`` (a sequence of ints) as a device ``[len(values)]``, without a wait for what the stream still has to do: a copy
    from pageable host memory has one. One number is a fill's argument; more go through pinned memory, which the allocator hands out
    again only after the copy."""
    if torch.device(device).type == "cpu":
        return torch.tensor(list(values), dtype=dtype)
    if len(values) == 1:
        return torch.full((1,), int(values[0]), dtype=dtype, device=device)
    return torch.tensor(list(values), dtype=dtype, pin_memory=True).to(device, non_blocking=True)
