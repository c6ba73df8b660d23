"""Release, retain and append of several layers at once equal the same
operations layer by layer, bit for bit (map, slab, free stack, templates, the
proven allocations), with layers that grow, layers that have room and a layer
on a paged map; a refused bank list changes no layer."""

from __future__ import annotations

import pytest
import torch

from copy_on_write_sdm_amd.allocator import PackedSDMCopyOnWriteState as State

pytestmark = pytest.mark.gpu

BANKS, SLOTS, WIDTH = 6, 32, 20


def _layers(device, banks, seed, pages=None, capacity=None):
    g = torch.Generator().manual_seed(seed)
    states = []
    for layer in range(3):
        m0 = torch.randn(2, SLOTS, WIDTH, generator=torch.Generator().manual_seed(layer))
        dense = torch.randn(banks, SLOTS, WIDTH, generator=g)
        active = torch.rand(banks, SLOTS, generator=g) < (0.1, 0.5, 0.9)[layer]
        state = State.from_dense_overlay(
            m0.to(device), dense.to(device), active.to(device),
            template_indices=(torch.arange(banks) % 2).to(device),
            capacity_rows=capacity, growth_quantum_rows=16,
            map_page_slots=4 if pages == layer else None)
        states.append(state)
    return states


def _same(a, b):
    for x, y in zip(a, b):
        with x._direct_form(keep=False), y._direct_form(keep=False):
            assert torch.equal(x.logical_to_physical, y.logical_to_physical)
        count = int(x.free_count)
        assert count == int(y.free_count)
        assert torch.equal(x.free_rows[:count], y.free_rows[:count])
        assert torch.equal(x.template_indices, y.template_indices)
        assert x.capacity_rows == y.capacity_rows and x.banks == y.banks
        assert (x.proven_maximum_additional_allocations
                == y.proven_maximum_additional_allocations)
        assert torch.equal(x.materialize_dense(), y.materialize_dense())
        x.validate_invariants()
        y.validate_invariants()


@pytest.mark.parametrize("pages", [None, 1])
@pytest.mark.parametrize("capacity", [None, 400])
def test_layers_equal_layer_by_layer(device, pages, capacity):
    a, b = (_layers(device, BANKS, 1, pages, capacity) for _ in range(2))
    gone = torch.tensor([4, 1], device=device)
    kept = torch.tensor([0, 2, 3, 5], device=device)
    rows = [int(n) for n in State.release_layers(a, [gone] * 3)]
    assert rows == [int(st.release(gone)) for st in b]
    _same(a, b)
    State.retain_banks_layers(a, [kept] * 3)
    for st in b:
        st.retain_banks(kept)
    _same(a, b)
    moved = State.append_banks_layers(a, _layers(device, 5, 2))
    assert moved == [st.append_banks_from(new) for st, new in zip(b, _layers(device, 5, 2))]
    _same(a, b)


def test_a_refused_list_changes_no_layer(device):
    a, b = (_layers(device, BANKS, 3) for _ in range(2))
    good, bad = torch.tensor([2], device=device), torch.tensor([2, 2], device=device)
    with pytest.raises(ValueError, match="invalid or duplicated"):
        State.release_layers(a, [good, good, bad])
    _same(a, b)
    with pytest.raises(ValueError, match="must be released before compaction"):
        State.retain_banks_layers(a, [good] * 3)
    _same(a, b)
