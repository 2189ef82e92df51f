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
