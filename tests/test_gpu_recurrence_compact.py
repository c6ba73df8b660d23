"""The dense-route recurrence where its compaction can go wrong
(csrc/recurrence.hip): tokens at the edge of what a compacted token holds
(8 and 9 nonzero write routes, 32 and 33 read routes), fully dense tokens and
tokens without a route, in sequences that cross the staged chunks and start
with either kind of token; slot
counts around the 64-slot segments; and values that are not finite.

The tolerance is the parity tests' (rtol 1e-4 / atol 2e-5, float64 oracle
sdm.py:464-529) scaled by the routes a token has: a sum of K float32 products
carries about K half-ulps, and the parity tests' routes hold 4, so a sum over
N dense routes is given N / 4 of it, at most 16 times (errors of random sign
grow with the root).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import copy_on_write_sdm_amd as cow
from oracle import serial

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-4, 2e-5


def _routes(rng, counts, slots):
    out = np.zeros(counts.shape + (slots,), np.float32)
    for at in np.ndindex(*counts.shape):
        k = min(int(counts[at]), slots)
        idx = rng.choice(slots, k, replace=False)
        w = rng.random(k).astype(np.float32) + 0.05
        out[at][idx] = w / max(1.0, w.sum())
    return out


def _inputs(batch, time, slots, width, seed, mixed=True):
    rng = np.random.default_rng(seed)
    writes = rng.choice([0, 1, 4, 8, 9, slots] if mixed else [1, 4, 8], (batch, time))
    reads = rng.choice([0, 1, 16, 32, 33, slots] if mixed else [1, 16, 32], (batch, time))
    gate = lambda: (1.0 / (1.0 + np.exp(-rng.standard_normal((batch, time))))).astype(np.float32)
    return dict(
        initial_memory=(rng.standard_normal((batch, slots, width)) * 0.5).astype(np.float32),
        write_routes=_routes(rng, writes, slots),
        values=rng.standard_normal((batch, time, width)).astype(np.float32),
        input_gate=gate(), erase_gate=gate(),
        forget_log_gate=(-rng.random((batch, time)) * 2.0).astype(np.float32),
        read_routes=_routes(rng, reads, slots))


def _oracle(a):
    with np.errstate(all="ignore"):
        return serial.serial_gated_delta_recurrence(
            a["initial_memory"], a["write_routes"], a["values"], a["input_gate"],
            a["forget_log_gate"], a["read_routes"], erase_gate=a["erase_gate"])


def _gpu(a, device):
    return {k: torch.from_numpy(v).to(device) for k, v in a.items()}


@pytest.mark.parametrize("batch,time,slots,width", [
    (9, 70, 33, 36), (2, 130, 64, 8), (128, 33, 64, 36), (128, 19, 33, 33), (3, 17, 65, 33), (1, 129, 256, 130), (2, 40, 257, 64),
    (2, 33, 1023, 40), (1, 20, 1024, 128)])
def test_mixed_tokens(device, batch, time, slots, width):
    print(f"mixed tokens B={batch} T={time} N={slots} D={width}", flush=True)
    a = _inputs(batch, time, slots, width, seed=slots)
    g = _gpu(a, device)
    readings, final, states = cow.sdm_recurrence(**g, return_states=True)
    scale = min(16.0, max(1.0, slots / 4))
    for got, want in zip((readings, final, states), _oracle(a)):
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=scale * RTOL, atol=scale * ATOL)
    assert torch.equal(states[:, -1], final)
    r2, m2 = cow.sdm_recurrence(**g)
    assert torch.equal(r2, readings) and torch.equal(m2, final)


@pytest.mark.parametrize("mixed", [False, True])
def test_a_token_depends_on_its_own_vectors_only(device, mixed):
    """Dense tokens put in among sparse ones change nothing before them."""

    a = _inputs(2, 45, 100, 40, seed=7, mixed=mixed)
    readings, _, states = cow.sdm_recurrence(**_gpu(a, device), return_states=True)
    t0 = 21
    b = {k: v.copy() for k, v in a.items()}
    b["write_routes"][:, t0:] = 0.01
    b["read_routes"][:, t0:] = 0.01
    r2, _, s2 = cow.sdm_recurrence(**_gpu(b, device), return_states=True)
    assert torch.equal(r2[:, :t0], readings[:, :t0])
    assert torch.equal(s2[:, :t0], states[:, :t0])


@pytest.mark.parametrize("slots,width", [(33, 64), (64, 130)])
def test_batch_size_changes_rounding_only(device, slots, width):
    """Up to 64 slots batch x width decides between two orders of summation:
    the same rows on either side of 4,096 agree within the tolerance."""

    print(f"batch sizes N={slots} D={width}", flush=True)
    a = _gpu(_inputs(4096 // width + 1, 21, slots, width, seed=slots, mixed=False), device)
    large = cow.sdm_recurrence(**a, return_states=True)
    small = cow.sdm_recurrence(**{k: v[:3].contiguous() for k, v in a.items()},
                               return_states=True)
    for x, y in zip(small, large):
        np.testing.assert_allclose(x.cpu().numpy(), y[:3].cpu().numpy(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("slots,width", [(70, 130), (300, 12)])
@pytest.mark.parametrize("first", [0, 1, 6, 7, 8, 15, 16, 31, 39])
def test_hand_over_at_the_first_dense_token(device, first, slots, width):
    """Sparse tokens, none with a route at first, up to token ``first`` and
    dense ones from there on: the oracle's results, and what comes before is
    the shorter sequence's, bit for bit."""

    print(f"hand over at {first} N={slots} D={width}", flush=True)
    a = _inputs(3, 40, slots, width, seed=first, mixed=False)
    a["write_routes"][:, 0] = a["read_routes"][:, 0] = 0.0
    rng = np.random.default_rng(first)
    a["write_routes"][1:, first] = _routes(rng, np.array([9, slots]), slots)
    a["write_routes"][0, first:] = _routes(rng, np.full(40 - first, 16), slots)
    a["read_routes"][0, first] = 0.0
    g = _gpu(a, device)
    readings, final, states = cow.sdm_recurrence(**g, return_states=True)
    scale = min(16.0, slots / 4)
    for got, want in zip((readings, final, states), _oracle(a)):
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=scale * RTOL, atol=scale * ATOL)
    assert torch.equal(states[:, -1], final)
    r2, m2 = cow.sdm_recurrence(**g)
    assert torch.equal(r2, readings) and torch.equal(m2, final)
    if first:
        part = {k: (v[:, :first].contiguous() if k != "initial_memory" else v)
                for k, v in g.items()}
        r0, m0 = cow.sdm_recurrence(**part)
        assert torch.equal(r0, readings[:, :first]) and torch.equal(m0, states[:, first - 1])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("planted", ["memory", "value", "weight", "read"])
def test_not_finite(device, mixed, planted):
    """The dense sums' NaN reach: zero routes times a value that is not
    finite are NaN too."""

    a = _inputs(2, 40, 70, 40, seed=11, mixed=mixed)
    if planted == "memory":
        a["initial_memory"][0, 69, 3] = np.inf
        a["initial_memory"][1, 0, 39] = np.nan
    elif planted == "value":
        a["values"][0, 19, 5] = np.inf
        a["values"][1, 33, 0] = np.nan
    elif planted == "weight":
        a["write_routes"][0, 18, 2] = np.nan
    else:
        a["read_routes"][1, 9, 2] = np.inf
    readings, final, states = cow.sdm_recurrence(**_gpu(a, device), return_states=True)
    for got, want in zip((readings, final, states), _oracle(a)):
        got = got.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = np.isfinite(want)
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
        np.testing.assert_allclose(got[ok], want[ok], rtol=16 * RTOL, atol=16 * ATOL)
