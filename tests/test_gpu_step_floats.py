"""16-bit weights, values and gates widened by the one-step kernel itself
(csrc/step_kernel.h, NARROW): bit for bit the step on inputs widened first
and its reading rounded by torch, at the edges of the kernel's shapes, with
mixed types, values at odd addresses, infinities and NaN, and shapes past the
kernel's, which are widened first."""

from __future__ import annotations

import pytest
import torch

import copy_on_write_sdm_amd as cow
from gpu_helpers import make_case, to_device

pytestmark = pytest.mark.gpu

H, F, B = torch.float16, torch.float32, torch.bfloat16
NAMES = ("write_weights", "values", "input_gate", "forget_log_gate", "read_weights")


@pytest.mark.parametrize("banks,slots,width,writes,reads", [
    (1, 16, 1, 1, 1), (5, 64, 63, 3, 15), (256, 32, 64, 4, 16), (7, 64, 100, 2, 16),
    (3, 64, 128, 4, 16), (2, 32, 256, 4, 8), (3, 64, 160, 4, 16), (4, 64, 128, 5, 17),
    (300, 16, 32, 2, 4)])
@pytest.mark.parametrize("types", [(B,) * 5, (H,) * 5, (F, B, H, F, B), (B, F, F, H, F)])
def test_narrow_inputs_equal_widened_ones(device, banks, slots, width, writes, reads, types):
    print(f"narrow step {(banks, slots, width, writes, reads)} {types}", flush=True)
    m0, steps = make_case(banks=banks, slots=slots, width=width, writes=writes, reads=reads,
                          steps=3, seed=width + banks)
    m0 = m0.to(device)
    states = [cow.PackedSDMCopyOnWriteState.allocate(m0, banks=banks,
                                                     capacity_rows=banks * slots)
              for _ in range(2)]
    tables = [m0.expand(banks, -1, -1).clone() for _ in range(2)]
    for s, inputs in enumerate(steps):
        x = to_device(inputs, device)
        if s == 2:
            x["values"][0, 0] = float("inf")
            x["values"][-1, -1] = float("nan")
            x["values"][0, width // 2] = 70000.0     # past float16's largest
        x = {k: (v.to(types[NAMES.index(k)]) if k in NAMES else v) for k, v in x.items()}
        values = x["values"]
        if s == 1:   # one element of offset
            odd = torch.empty(values.numel() + 1, dtype=values.dtype, device=device)[1:]
            x["values"] = odd.view_as(values).copy_(values)
        wide = {k: (v.float() if k in NAMES else v) for k, v in x.items()}
        got, got_diag = cow.packed_sdm_cow_step(states[0], **x)
        want, want_diag = cow.packed_sdm_cow_step(states[1], **wide)
        dense = cow.dense_sdm_sparse_step(tables[0], **x)
        cow.dense_sdm_sparse_step(tables[1], **wide)
        want = want.to(values.dtype)
        for reading in (got, dense):
            assert reading.dtype == values.dtype
            assert torch.equal(reading.isnan(), want.isnan())
            assert torch.equal(reading.nan_to_num(7.0), want.nan_to_num(7.0))
        assert torch.equal(got_diag.first_touches_by_sequence,
                           want_diag.first_touches_by_sequence)
    assert torch.equal(states[0].logical_to_physical, states[1].logical_to_physical)
    for a, b in ((states[0].materialize_dense(), states[1].materialize_dense()), tables):
        assert torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0))


@pytest.mark.parametrize("name", NAMES)
def test_a_refused_step_takes_no_pages(device, name):
    """Weights, values and gates that no step takes are refused before a paged
    map is given room for the step."""

    print(f"refused step, {name} in float64", flush=True)
    m0, steps = make_case(banks=4, slots=64, width=32, writes=2, reads=4, steps=1, seed=1)
    state = cow.PackedSDMCopyOnWriteState.allocate(m0.to(device), banks=4, capacity_rows=256,
                                                   map_page_slots=16)
    before = state.paged_map.pages_bound, state.paged_map.capacity
    x = to_device(steps[0], device)
    x[name] = x[name].double()
    with pytest.raises(ValueError, match="float32 weights, values and gates"):
        cow.packed_sdm_cow_step(state, **x)
    assert (state.paged_map.pages_bound, state.paged_map.capacity) == before
