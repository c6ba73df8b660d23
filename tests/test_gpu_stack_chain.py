"""A run of SDM layers without a tail between them (one chain of launches,
decode_sdm_layers_controller) against the same layers one by one: tokens and
states (maps, slabs, free stacks, growth, proofs) bit for bit over several
tokens, for layers alike and unlike (heads, slots, route counts: every form
of the route selection), one to four of them, few and many tokens, slabs that
grow on the way and slabs that are proven, and a paged layer that splits the
run."""

from __future__ import annotations

import pytest
import torch

import copy_on_write_sdm_amd as cow
from controller_cases import make_layer
from gpu_helpers import assert_states_identical

pytestmark = pytest.mark.gpu

WIDTH = 128
ALIKE = [(1, 256, 16, 4)] * 4                       # (heads, slots, reads, writes)
UNLIKE = [(1, 64, 4, 1), (4, 256, 16, 4), (2, 1024, 24, 6), (1, 4225, 16, 4)]
WIDENING = [(1, 256, 16, 4), (1, 64, 8, 2), (4, 256, 16, 4)]


def _stack(device, shapes, batch, grows, paged):
    ctrls, stacks = [], ([], [])
    for i, (heads, slots, reads, writes) in enumerate(shapes):
        layer = make_layer(WIDTH, slots=slots, reads=reads, writes=writes, heads=heads, seed=i,
                           dtype=torch.float32)
        ctrls.append(cow.SDMController.from_module(layer, device=device))
        g = torch.Generator().manual_seed(50 + i)
        m0 = (torch.randn(heads, slots, WIDTH // heads, generator=g) * 0.3).to(device)
        banks = batch * heads
        quantum = banks * writes + 3
        for states in stacks:
            st = cow.PackedSDMCopyOnWriteState.allocate(
                m0, banks=banks, capacity_rows=quantum if grows else banks * slots,
                template_indices=torch.arange(heads, device=device).repeat(batch),
                growth_quantum_rows=quantum if grows else 0,
                map_page_slots=16 if i == paged else None)
            st.capacity_is_proven = True
            states.append(st)
    return ctrls, *stacks


def _decode_state(states, layout, batch, device):
    return cow.FaithfulSDMDecodeState(
        layout=layout, position=0, capacity=16, activation_dtype=torch.float32,
        active_sequences=torch.ones(batch, dtype=torch.bool, device=device),
        sdm_layer_positions=tuple(i for i, k in enumerate(layout) if k == "B"),
        sdm_states=tuple(states),
        dense_keys=tuple(torch.zeros(batch, 1, 16, 4, device=device)
                         for _ in range(layout.count("A"))),
        dense_values=tuple(torch.zeros(batch, 1, 16, 4, device=device)
                           for _ in range(layout.count("A"))))


@pytest.mark.parametrize("shapes,layout,batch,grows,paged", [
    (ALIKE[:1], "B", 3, True, None),
    (ALIKE[:2], "BB", 1, False, None),
    (ALIKE, "BBBB", 64, True, None),
    (ALIKE, "BBABB", 5, True, None),
    (UNLIKE, "BBBB", 1, True, None),
    (UNLIKE, "BBBB", 64, False, None),
    (WIDENING, "BBB", 16, True, None),
    (WIDENING, "BBB", 300, True, None),
    (WIDENING, "BBB", 1100, False, None),
    (ALIKE, "BBBB", 16, True, 2),
])
def test_chain_equals_layer_by_layer(device, shapes, layout, batch, grows, paged):
    print(f"stack chain {shapes} {layout} B={batch} grows={grows} paged={paged}", flush=True)
    ctrls, chained, single = _stack(device, shapes, batch, grows, paged)
    state = _decode_state(chained, layout, batch, device)
    g = torch.Generator().manual_seed(7)
    for step in range(4):
        x = torch.randn(batch, 1, WIDTH, generator=g).to(device)
        got = cow.decode_faithful_sdm_stack(
            layout, ctrls, x, state, attention_decode=lambda layer, t, k, v, p: t * 0.5 + 0.1)
        want, at = x, 0
        for kind in layout:
            if kind == "A":
                want = want * 0.5 + 0.1
                continue
            want = want + cow.decode_sdm_layer_controller(ctrls[at], want, single[at])
            at += 1
        assert torch.equal(got, want), step
    for a, b in zip(chained, single):
        assert_states_identical(a, b)
    if grows:
        assert sum(st.growth_events for st in chained) > 0
