"""Values that are not finite, and sums that overflow, in the token-serial
recurrences: the same rows and readings are NaN, +inf and -inf as in the
dense float32 sums (sdm.py:464-529), where a zero route times such a row or
delta is NaN and a row that a route writes is not, at any token (the last of
a sequence among them, where the kernels' chunks go on past it), and the other
columns and the earlier tokens keep the bits that they have without.

Tolerance of what stays finite: rtol 1e-4 / atol 2e-5, the parity tests'."""

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
COLUMN = 5
PLANTED = ["memory", "written memory", "value", "last value", "gate", "weight", "last weight",
           "overflow", "last overflow", "last overflow, unread"]


def _dense_sums(start, wr, values, gate, forget, rr, erase):
    """The recurrence in float32, every sum over all rows."""

    memory, readings, states = start.copy(), [], []
    with np.errstate(all="ignore"):
        for t in range(wr.shape[1]):
            w, r = wr[:, t, :, None], rr[:, t, :, None]
            memory = np.where(w != 0, memory * np.exp(forget[:, t])[:, None, None], memory)
            delta = (gate[:, t, None] * values[:, t]
                     - erase[:, t, None] * (w * memory).sum(axis=1))
            memory = memory + w * delta[:, None]
            readings.append((r * memory).sum(axis=1))
            states.append(memory.copy())
    return np.stack(readings, axis=1), memory, np.stack(states, axis=1)


def _assert_same(got, want):
    got = got.cpu().numpy()
    assert want.dtype == np.float32
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert np.isfinite(got[ok]).all()
    np.testing.assert_allclose(got[ok], want[ok], rtol=RTOL, atol=ATOL)


def _case(time, slots, width, writes, reads, seed):
    rng = np.random.default_rng(seed)
    idx = np.argsort(rng.random((2, time, slots)), axis=2)
    ww = rng.random((time, writes)).astype(np.float32) + 0.1
    rw = rng.random((time, reads)).astype(np.float32) + 0.1
    return dict(
        m0=(0.5 * rng.standard_normal((slots, width))).astype(np.float32),
        write_indices=idx[0, :, :writes], write_weights=ww / ww.sum(1, keepdims=True),
        read_indices=idx[1, :, :reads], read_weights=rw / rw.sum(1, keepdims=True),
        values=rng.standard_normal((time, width)).astype(np.float32),
        input_gate=(0.2 + 0.6 * rng.random(time)).astype(np.float32),
        forget_log_gate=(-2 * rng.random(time)).astype(np.float32))


def _plant(a, planted):
    """One fault in column COLUMN of ``a`` (the gate's and the weight's are in
    every column); the token it is at."""

    time = len(a["values"])
    t = 0 if "memory" in planted else time - 1 if "last" in planted else time // 3
    row = a["write_indices"][t, 0]
    if planted == "memory":
        a["m0"][(a["write_indices"][0, -1] + 1) % len(a["m0"]), COLUMN] = np.inf
    elif planted == "written memory":
        a["m0"][row, COLUMN] = -np.inf
    elif "value" in planted:
        a["values"][t, COLUMN] = -np.inf
    elif planted == "gate":
        a["input_gate"][t] = np.inf
    elif "weight" in planted:
        a["write_weights"][t, 0] = np.nan
    else:
        # the first written row holds 3e38 until token t adds 0.5 * (v - 0.5 * 3e38)
        a["m0"][row, COLUMN] = 3e38
        a["write_weights"][:t][a["write_indices"][:t] == row] = 0.0
        a["read_weights"][:t][a["read_indices"][:t] == row] = 0.0
        a["write_weights"][t] = 0.0
        a["write_weights"][t, 0] = 0.5
        a["input_gate"][t], a["forget_log_gate"][t] = 1.0, 0.0
        a["values"][t, COLUMN] = 3.4e38
        seen = a["read_indices"][t] == row
        if "unread" in planted:
            a["read_weights"][t][seen] = 0.0
        elif not seen.any():
            a["read_indices"][t, 0] = row
    return t


@pytest.mark.parametrize("planted", PLANTED)
@pytest.mark.parametrize("time,slots,width,writes,reads", [
    (1, 64, 40, 4, 8), (20, 64, 40, 4, 16), (64, 100, 130, 9, 24), (16, 12, 6, 12, 12)])
def test_route_recurrence(device, time, slots, width, writes, reads, planted):
    print(f"route recurrence T={time} N={slots} W={writes} {planted}", flush=True)
    a = _case(time, slots, width, writes, reads, seed=time)
    x = lambda: SimpleNamespace(**{k: torch.from_numpy(v.copy()).to(device)
                                   for k, v in a.items() if k != "m0"})
    m0 = lambda: torch.from_numpy(a["m0"].copy()).to(device)[None]
    before = route_recurrence(m0(), x(), 1, time)
    t = _plant(a, planted)
    readings, final = route_recurrence(m0(), x(), 1, time)
    wr, rr = (serial.dense_routes(a[f"{k}_indices"][None], a[f"{k}_weights"][None],
                                  slots).astype(np.float32) for k in ("write", "read"))
    want_r, want_m, _ = _dense_sums(a["m0"][None], wr, a["values"][None], a["input_gate"][None],
                                    a["forget_log_gate"][None], rr, a["input_gate"][None])
    _assert_same(readings[None], want_r)
    _assert_same(final, want_m)
    if "overflow" not in planted:
        assert torch.equal(readings[:t], before[0][:t])
    if "memory" in planted or "value" in planted:
        others = [c for c in range(width) if c != COLUMN]
        assert torch.equal(readings[:, others], before[0][:, others])
        assert torch.equal(final[:, :, others], before[1][:, :, others])


@pytest.mark.parametrize("planted", PLANTED)
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("time,slots,width,writes,reads", [
    (1, 70, 40, 4, 8), (20, 70, 33, 4, 16), (48, 100, 130, 8, 24), (17, 300, 12, 4, 32),
    (20, 32, 16, 4, 8)])
def test_dense_route_recurrence(device, time, slots, width, writes, reads, mixed, planted):
    """``mixed``: every third token has a route to every row."""

    print(f"recurrence T={time} N={slots} W={writes} mixed={mixed} {planted}", flush=True)
    a = _case(time, slots, width, writes, reads, seed=time + slots)

    def inputs():
        routes = {}
        for k in ("write", "read"):
            x = serial.dense_routes(a[f"{k}_indices"][None], a[f"{k}_weights"][None],
                                    slots).astype(np.float32)
            if mixed:
                x[:, 1:-1:3] += np.float32(0.2 / slots)
            routes[f"{k}_routes"] = x
        return dict(initial_memory=a["m0"][None], values=a["values"][None],
                    input_gate=a["input_gate"][None], erase_gate=a["input_gate"][None],
                    forget_log_gate=a["forget_log_gate"][None], **routes)

    def run(x):
        return cow.sdm_recurrence(**{k: torch.from_numpy(v.copy()).to(device)
                                     for k, v in x.items()}, return_states=True)

    before = run(inputs())
    t = _plant(a, planted)
    if mixed and planted == "overflow":
        # the row's 3e38 would reach the others through the tokens of all rows
        a["m0"][a["write_indices"][t, 0], COLUMN] = 0.0
        a["values"][t, COLUMN] = np.inf
    x = inputs()
    if mixed and "last overflow" in planted:
        row = a["write_indices"][t, 0]
        x["write_routes"][:, :t, row] = x["read_routes"][:, :t, row] = 0.0
    readings, final, states = run(x)
    want = _dense_sums(x["initial_memory"], x["write_routes"], x["values"], x["input_gate"],
                       x["forget_log_gate"], x["read_routes"], x["erase_gate"])
    for got, expected in zip((readings, final, states), want):
        _assert_same(got, expected)
    r2, m2 = cow.sdm_recurrence(**{k: torch.from_numpy(v.copy()).to(device)
                                   for k, v in x.items()})
    assert torch.equal(r2.nan_to_num(1.5), readings.nan_to_num(1.5))
    assert torch.equal(m2.nan_to_num(1.5), final.nan_to_num(1.5))
    if "overflow" not in planted:
        assert torch.equal(readings[:, :t], before[0][:, :t])
        assert torch.equal(states[:, :t], before[2][:, :t])
    if "memory" in planted or "value" in planted:
        others = [c for c in range(width) if c != COLUMN]
        for got, same in zip((readings, final, states), before):
            assert torch.equal(got[..., others], same[..., others])
