"""Host-side checks of the stack decode (decode_faithful_sdm_stack,
inference.py:601-669) that run before any device work, and the dense K/V
cache write of one decode token (decode_with_cache, model.py:138-162), on
the CPU: every refusal keeps the reference's message, and a refused call
changes neither the positions nor the caches."""

from __future__ import annotations

import math
from types import SimpleNamespace

import pytest
import torch

import copy_on_write_sdm_amd as cow
from copy_on_write_sdm_amd import _native as nat
from copy_on_write_sdm_amd import controller as controller_module


def _state(*, layout="BAB", batch=3, position=5, capacity=8, positions=None,
           sdm=2, dense=1, layer_positions=None):
    keys = tuple(torch.zeros(batch, 2, capacity, 4) for _ in range(dense))
    return cow.FaithfulSDMDecodeState(
        layout=layout, position=position, capacity=capacity, activation_dtype=torch.float32,
        active_sequences=torch.ones(batch, dtype=torch.bool),
        sdm_layer_positions=(layer_positions if layer_positions is not None
                             else tuple(i for i, k in enumerate(layout) if k == "B")),
        sdm_states=tuple(object() for _ in range(sdm)), dense_keys=keys,
        dense_values=tuple(k.clone() for k in keys), positions=positions)


CONTROLLERS = [SimpleNamespace(width=16), SimpleNamespace(width=16)]


def _decode(state, tokens=None, layout="BAB", controllers=CONTROLLERS, **kw):
    tokens = torch.zeros(state.batch, 1, 16) if tokens is None else tokens
    kw.setdefault("attention_decode", lambda *a: a[1])
    return cow.decode_faithful_sdm_stack(layout, controllers, tokens, state, **kw)


def test_refusals_keep_the_reference_messages():
    with pytest.raises(ValueError, match=r"decode tokens must be \[3,1,16\]"):
        _decode(_state(), torch.zeros(3, 2, 16))
    with pytest.raises(ValueError, match=r"decode tokens must be \[3,1,16\]"):
        _decode(_state(), torch.zeros(2, 1, 16))
    with pytest.raises(ValueError, match="layout does not match the stack"):
        _decode(_state(layout="BBA", layer_positions=(0, 1)))
    with pytest.raises(ValueError, match="do not match state device and dtype"):
        _decode(_state(), torch.zeros(3, 1, 16, dtype=torch.float64))
    with pytest.raises(ValueError, match="reached its fixed capacity"):
        _decode(_state(position=8, capacity=8))
    with pytest.raises(ValueError, match="reached its fixed capacity"):
        _decode(_state(position=7, positions=torch.tensor([3, 8, 7])))
    released = _state()
    released.active_sequences[1] = False
    with pytest.raises(ValueError, match="released requests must be removed"):
        _decode(released)
    with pytest.raises(ValueError, match="decode state does not match the stack"):
        _decode(_state(sdm=1))
    with pytest.raises(ValueError, match="decode state does not match the stack"):
        _decode(_state(dense=0))
    with pytest.raises(ValueError, match="decode state does not match the stack"):
        _decode(_state(), controllers=CONTROLLERS[:1])
    with pytest.raises(ValueError, match="ordering is inconsistent"):
        _decode(_state(layer_positions=(2, 0)))
    with pytest.raises(ValueError, match="attention_decode"):
        _decode(_state(), attention_decode=None)
    with pytest.raises(ValueError, match="share its width"):
        _decode(_state(), controllers=[SimpleNamespace(width=16), SimpleNamespace(width=8)])


def test_refused_call_leaves_positions_alone():
    positions = torch.tensor([3, 8, 7])
    state = _state(position=8, positions=positions)
    with pytest.raises(ValueError, match="fixed capacity"):
        _decode(state)
    assert positions.tolist() == [3, 8, 7] and state.position == 8


def test_attention_only_stack_advances_positions():
    """A stack without SDM layers runs only the caller's attention and moves
    the shared position, or every request's own, one token on."""

    seen = []

    def attention(layer, tokens, key_cache, value_cache, position):
        seen.append((layer, position if isinstance(position, int) else position.tolist()))
        return tokens + 1

    state = _state(layout="AA", sdm=0, dense=2, position=2)
    out = cow.decode_faithful_sdm_stack("AA", [], torch.zeros(3, 1, 4), state,
                                        attention_decode=attention)
    assert torch.equal(out, torch.full((3, 1, 4), 2.0))
    assert seen == [(0, 2), (1, 2)] and state.position == 3 and state.positions is None
    seen.clear()
    positions = torch.tensor([1, 6, 4])
    state = _state(layout="AA", sdm=0, dense=2, position=6, positions=positions)
    cow.decode_faithful_sdm_stack("AA", [], torch.zeros(3, 1, 4), state,
                                  attention_decode=attention)
    assert seen == [(0, [1, 6, 4]), (1, [1, 6, 4])]
    assert state.positions.tolist() == [2, 7, 5] and state.position == 7


def test_dense_cache_write_at_shared_and_own_positions():
    caches = torch.zeros(3, 2, 6, 4), torch.zeros(3, 2, 6, 4)
    key = torch.arange(24, dtype=torch.float32).reshape(3, 2, 1, 4) + 1
    cow.write_dense_cache(*caches, key, -key, position=2)
    assert torch.equal(caches[0][:, :, 2:3], key) and torch.equal(caches[1][:, :, 2:3], -key)
    assert caches[0][:, :, [0, 1, 3, 4, 5]].abs().sum() == 0
    cow.write_dense_cache(*caches, 2 * key, -2 * key, position=torch.tensor([0, 5, 3]))
    for b, p in enumerate((0, 5, 3)):
        assert torch.equal(caches[0][b, :, p], 2 * key[b, :, 0])
        assert torch.equal(caches[1][b, :, p], -2 * key[b, :, 0])
    with pytest.raises(ValueError, match="positions are invalid"):
        cow.write_dense_cache(*caches, key, key, position=torch.tensor([0, 1]))
    with pytest.raises(ValueError, match="cache is invalid"):
        cow.write_dense_cache(caches[0], caches[1][:, :, :5], key, key, position=1)
    with pytest.raises(ValueError, match="cache is invalid"):
        cow.write_dense_cache(*caches, key.expand(3, 2, 2, 4), key.expand(3, 2, 2, 4),
                              position=1)


class _Launches:
    """The library's entries of a chain of SDM layers, each recorded as the
    byte ranges that it reads and writes."""

    def __init__(self):
        self.launches = []   # (ranges read, ranges written)

    @staticmethod
    def _prepared(c, batch, args):
        normalized, read_keys, write_keys, values, gate, forget, _, _, rw, ri, ww, wi = args
        banks = batch * c.memory_heads
        reads, writes = c.route_counts()
        sizes = ((normalized, batch * c.width), (read_keys, banks * c.key_width_per_head),
                 (write_keys, banks * c.key_width_per_head), (values, batch * c.width),
                 (gate, banks), (forget, banks), (rw, banks * reads), (ri, 2 * banks * reads),
                 (ww, banks * writes), (wi, 2 * banks * writes))
        return [(at, at + 4 * n) for at, n in sizes]

    @staticmethod
    def _tokens(batch, c, *pointers):
        return [(at, at + 4 * batch * c.width) for at in pointers]

    def cowsdm_controller_prepare_routes(self, c, tokens, batch, *rest):
        self.launches.append((self._tokens(batch, c, tokens),
                              self._prepared(c, batch, rest[:-1])))
        return 0

    def cowsdm_packed_step(self, layer, shape, stream):
        banks, floats = shape.banks, shape.banks * shape.width
        read = ((layer.write_indices, 2 * banks * shape.writes),
                (layer.write_weights, banks * shape.writes), (layer.step_values, floats),
                (layer.input_gate, banks), (layer.forget_log_gate, banks),
                (layer.read_indices, 2 * banks * shape.reads),
                (layer.read_weights, banks * shape.reads))
        self.launches.append(([(at, at + 4 * n) for at, n in read],
                              [(layer.output, layer.output + 4 * floats)]))
        return 0

    def cowsdm_controller_finish_residual(self, c, normalized, reading, batch, out, residual,
                                          total, stream):
        self.launches.append((self._tokens(batch, c, normalized, reading, residual),
                              self._tokens(batch, c, out, total)))
        return 0

    def cowsdm_controller_finish_prepare_routes(self, c, normalized, reading, batch, out,
                                                residual, total, following, *rest):
        self.launches.append((self._tokens(batch, c, normalized, reading, residual),
                              self._tokens(batch, c, out, total)
                              + self._prepared(following, batch, rest[:-1])))
        return 0


@pytest.mark.parametrize("batch", [1, 16, 64])
@pytest.mark.parametrize("shapes", [
    ((1, 256, 16, 4), (1, 256, 16, 4), (4, 256, 16, 4)),      # (heads, slots, reads, writes)
    ((1, 64, 4, 1), (4, 1024, 32, 8), (2, 1024, 16, 4), (1, 64, 4, 1), (8, 256, 16, 4)),
    ((2, 256, 16, 4),) * 4])
def test_chained_layers_share_no_bytes_within_a_launch(monkeypatch, shapes, batch):
    """decode_sdm_layers_controller's launches, layers alike or not: what a
    launch writes overlaps nothing else that it reads or writes (its
    workgroups are not ordered), and what it reads was last written whole, by
    one launch."""

    width = 128
    library = _Launches()
    monkeypatch.setattr(nat, "lib", lambda: library)
    monkeypatch.setattr(nat, "stream_handle", lambda device: 0)
    monkeypatch.setattr(controller_module, "_check_tokens", lambda c, tokens: tokens.shape[0])
    controllers, states = [], []
    for heads, slots, reads, writes in shapes:
        root = math.isqrt(slots)
        c = SimpleNamespace(
            width=width, memory_heads=heads, head_width=width // heads, reads=reads,
            writes=writes, key_width_per_head=2 * root,
            route_counts=lambda r=reads, w=writes, n=root: (min(r, min(r, n) ** 2),
                                                            min(w, min(w, n) ** 2)))
        c.c_struct = lambda c=c: c
        controllers.append(c)
        empty = torch.empty(1)
        states.append(SimpleNamespace(
            banks=batch * heads, width=width // heads, slots=slots, values=empty,
            growth_quantum_rows=0, shared_initial_memory=empty, template_indices=empty,
            logical_to_physical=empty, free_rows=empty, free_count=empty, overflow_flag=empty,
            ensure_scratch=lambda: torch.empty(1), capacity_rows=1))
    tokens = torch.zeros(batch, 1, width)
    result = controller_module.decode_sdm_layers_controller(controllers, states, tokens)
    assert len(library.launches) == 2 * len(shapes) + 1
    held = [(tokens.data_ptr(), tokens.data_ptr() + 4 * tokens.numel())]   # whole, as written
    for read, written in library.launches:
        for i, (low, high) in enumerate(written):
            for other_low, other_high in read + written[:i] + written[i + 1:]:
                assert high <= other_low or other_high <= low
        for low, high in read:
            assert any(a <= low and high <= b for a, b in held)
        held = [(a, b) for a, b in held
                if all(high <= a or b <= low for low, high in written)] + written
    assert (result.data_ptr(), result.data_ptr() + 4 * result.numel()) in held
