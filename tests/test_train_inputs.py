"""Which training calls the one-call layer takes: adapters whose shapes the library cannot read by one
rank go through the per-projection functions."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from experts4bit_qlora_amd import train

E, R, HID, INTER, T, K = 4, 8, 128, 64, 6, 2


def _module(**change):
    shapes = dict(gate_up_lora_A=(E, R, HID), gate_up_lora_B=(E, 2 * INTER, R), down_lora_A=(E, R, INTER),
                  down_lora_B=(E, HID, R))
    shapes.update(change)
    base = SimpleNamespace(act_fn=F.silu, has_gate=True, num_experts=E, _gate_up_shape=(2 * INTER, HID),
                           _down_shape=(HID, INTER))
    return SimpleNamespace(base=base, **{k: torch.zeros(s) for k, s in shapes.items()})


def _inputs(mod):
    return train._layer_inputs(mod, torch.zeros(T, HID, dtype=torch.bfloat16), torch.zeros(T, K, dtype=torch.int64),
                               torch.zeros(T, K))


def test_matching_adapters_take_the_layer():
    assert _inputs(_module()) is not None


@pytest.mark.parametrize("change", [
    dict(down_lora_A=(E, 4, INTER), down_lora_B=(E, HID, 4)),   # a second rank
    dict(down_lora_A=(E, 4, INTER)), dict(gate_up_lora_B=(E, 2 * INTER, 4)), dict(gate_up_lora_A=(E - 1, R, HID)),
    dict(gate_up_lora_A=(E * R, HID)), dict(down_lora_B=(E, HID // 2, R)), dict(gate_up_lora_A=(E, R, HID // 2)),
])
def test_other_adapter_shapes_do_not(change):
    assert _inputs(_module(**change)) is None
