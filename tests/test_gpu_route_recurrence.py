"""GPU parity of the sparse-route recurrence of a layer's prefill
(csrc/route_recurrence.hip) against ``oracle.serial`` (float64,
sdm.py:464-529) and the dense-route kernel, at the sizes where its layout
turns: chunks of 16, 32 and 64 tokens, the groups of 8 tokens and 8 lanes,
partial column blocks, one to four routes per lane, the largest table.

Tolerance rtol 1e-4 / atol 2e-5 as for the dense-route kernel: both sum in
float32, in an order of their own."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

import copy_on_write_sdm_amd as cow
from copy_on_write_sdm_amd.recurrence import route_recurrence
from oracle import serial

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-4, 2e-5


def _case(batch, time, heads, slots, width, writes, reads, seed):
    rng = np.random.default_rng(seed)
    rows = batch * time * heads

    def routes(k):
        return np.argsort(rng.random((rows, slots)), axis=1)[:, :k].astype(np.int64)

    ww = rng.random((rows, writes)).astype(np.float32)
    ww[rng.random((rows, writes)) < 0.1] = 0.0      # a zero route leaves its row alone
    rw = rng.random((rows, reads)).astype(np.float32)
    return dict(
        m0=(rng.standard_normal((heads, slots, width)) * 0.5).astype(np.float32),
        write_indices=routes(writes), write_weights=ww / (ww.sum(1, keepdims=True) + 1e-3),
        read_indices=routes(reads), read_weights=rw / rw.sum(1, keepdims=True),
        values=rng.standard_normal((rows, width)).astype(np.float32),
        input_gate=(1 / (1 + np.exp(-rng.standard_normal(rows)))).astype(np.float32),
        forget_log_gate=(-2 * rng.random(rows)).astype(np.float32))


def _run(a, batch, time, device):
    x = {k: torch.from_numpy(v.astype(np.float32) if v.dtype == np.float64 else v).to(device)
         for k, v in a.items()}
    m0 = x.pop("m0")
    return route_recurrence(m0, SimpleNamespace(**x), batch, time)


def _by_bank(v, batch, time, heads):
    v = v.reshape(batch, time, heads, *v.shape[1:])
    return np.ascontiguousarray(np.swapaxes(v, 1, 2)).reshape(batch * heads, time, *v.shape[3:])


@pytest.mark.parametrize("batch,time,heads,slots,width,writes,reads", [
    (1, 1, 1, 1, 1, 1, 1),
    (2, 63, 1, 256, 128, 4, 16),
    (9, 64, 1, 64, 32, 8, 8),
    (1, 65, 2, 100, 33, 9, 17),
    (3, 130, 1, 256, 40, 1, 9),
    (1, 71, 4, 1024, 100, 16, 32),
    (1, 50, 1, 1023, 128, 32, 32),
    (2, 17, 3, 36, 7, 17, 3),
])
def test_route_recurrence_matches_oracle(device, batch, time, heads, slots, width, writes, reads):
    print(f"route recurrence {(batch, time, heads, slots, width, writes, reads)}", flush=True)
    a = _case(batch, time, heads, slots, width, writes, reads, seed=time + slots)
    readings, final = _run(a, batch, time, device)
    banks = {k: _by_bank(v, batch, time, heads) for k, v in a.items() if k != "m0"}
    wr = serial.dense_routes(banks["write_indices"], banks["write_weights"], slots)
    rr = serial.dense_routes(banks["read_indices"], banks["read_weights"], slots)
    start = np.broadcast_to(a["m0"][None], (batch, heads, slots, width)).reshape(-1, slots, width)
    want_r, want_m, _ = serial.serial_gated_delta_recurrence(
        start, wr, banks["values"], banks["input_gate"], banks["forget_log_gate"], rr,
        erase_gate=banks["input_gate"])
    got = _by_bank(readings.cpu().numpy(), batch, time, heads)
    np.testing.assert_allclose(got, want_r, rtol=RTOL, atol=ATOL)
    np.testing.assert_allclose(final.cpu().numpy(), want_m, rtol=RTOL, atol=ATOL)
    # rows that no route writes keep their initial memory bit for bit
    same = (wr == 0).all(axis=1)
    assert np.array_equal(final.cpu().numpy()[same], start[same].astype(np.float32))


@pytest.mark.parametrize("where", ["memory", "value", "last value", "gate"])
def test_non_finite_values_spread_as_in_the_dense_sums(device, where):
    """A zero route times a non-finite row is NaN in the dense sums, so every
    later reading of the column is; the finite columns do not change."""

    batch, time, slots, width = 1, 20, 64, 40
    a = _case(batch, time, 1, slots, width, 4, 8, seed=3)
    if where == "memory":
        a["m0"][0, 5, 11] = np.inf
    elif where == "value":
        a["values"][7, 33] = -np.inf
    elif where == "last value":
        a["values"][-1, 2] = np.nan
    else:
        a["input_gate"][9] = np.inf
    readings, final = _run(a, batch, time, device)
    dense = {k: torch.from_numpy(serial.dense_routes(
        a[f"{k}_indices"][None], a[f"{k}_weights"][None], slots).astype(np.float32)).to(device)
        for k in ("write", "read")}
    x = {k: torch.from_numpy(a[k])[None].to(device)
         for k in ("values", "input_gate", "forget_log_gate")}
    want_r, want_m = cow.gated_delta_recurrence(
        torch.from_numpy(a["m0"]).to(device), dense["write"], x["values"], x["input_gate"],
        x["forget_log_gate"], dense["read"])
    for got, want in ((readings[None], want_r), (final, want_m)):
        got, want = got.cpu().numpy(), want.cpu().numpy()
        assert np.array_equal(np.isfinite(got), np.isfinite(want))
        ok = np.isfinite(want)
        np.testing.assert_allclose(got[ok], want[ok], rtol=RTOL, atol=ATOL)
