"""The controller's matrix-core projections (csrc/controller.hip) at the edges
of their tiles: widths around the groups of 16 inputs (below one, odd, more
than a chunk of weights), batches around the tiles of 16 tokens and each
kernel form's range, inputs at odd addresses.  Against oracle/controller.py
within test_gpu_controller.py's tolerances on the first and last tokens, and
a token's outputs do not depend on the batch it is in, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from controller_cases import make_layer, params_of
from copy_on_write_sdm_amd import controller as ctl
from oracle import controller as octl

pytestmark = pytest.mark.gpu

# 1 .. 256 tokens a workgroup each, tiles of one row a lane to 512, two rows
# above, two tiles of tokens from 8,192 on (where LDS allows)
@pytest.mark.parametrize("width,heads,slots", [
    (6, 2, 4), (16, 1, 16), (33, 1, 25), (50, 2, 64), (128, 1, 256), (132, 4, 100),
    (272, 1, 64), (1000, 4, 16)])
@pytest.mark.parametrize("batch", [1, 17, 257, 515, 8207])
def test_tiles_match_oracle_and_any_batch(device, width, heads, slots, batch):
    print(f"controller tiles width={width} H={heads} N={slots} B={batch}", flush=True)
    layer = make_layer(width, slots=slots, reads=min(8, slots), writes=min(4, slots),
                       heads=heads, seed=width + batch, dtype=torch.float32)
    c = ctl.SDMController.from_module(layer, device=device)
    g = torch.Generator(device=device).manual_seed(batch)
    x = torch.randn(batch, 1, width, generator=g, device=device)
    step = ctl.prepare_sdm_step(c, x)
    reading = torch.randn(batch * heads, width // heads, generator=g, device=device)
    out = ctl.finish_sdm_step(c, step, reading)
    inp = step.inputs

    ends = list(range(min(batch, 3))) + ([batch - 2, batch - 1] if batch > 3 else [])
    rows = [b * heads + h for b in ends for h in range(heads)]
    p = params_of(layer)
    want = octl.prepare(p, x[ends].cpu().numpy())

    def close(got, wanted, rtol=1e-4, atol=2e-5):
        np.testing.assert_allclose(got.cpu().numpy(), wanted, rtol=rtol, atol=atol)

    close(step.normalized[ends], want["normalized"], 1e-5, 1e-5)
    close(inp.values[rows], want["values"])
    close(inp.input_gate[rows], want["input_gate"])
    close(inp.forget_log_gate[rows], want["forget_log_gate"])
    close(out[ends], octl.finish(p, step.normalized[ends].cpu().numpy().astype(np.float64),
                                 reading[rows].cpu().numpy().astype(np.float64)))

    # the last tokens alone, from an odd address
    some = slice(max(0, batch - 5), batch)
    few = x[some]
    odd = torch.empty(few.numel() + 1, device=device)[1:].view_as(few).copy_(few)
    again = ctl.prepare_sdm_step(c, odd)
    banks = slice(some.start * heads, batch * heads)
    assert torch.equal(again.normalized, step.normalized[some])
    for name in ("values", "input_gate", "forget_log_gate", "read_indices", "read_weights",
                 "write_indices", "write_weights"):
        assert torch.equal(getattr(again.inputs, name), getattr(inp, name)[banks]), name
    assert torch.equal(ctl.finish_sdm_step(c, again, reading[banks]), out[some])


@pytest.mark.parametrize("width,heads,slots,reads,batch", [
    (128, 1, 256, 16, 4096), (128, 1, 256, 16, 4097), (64, 4, 256, 24, 1024),
    (64, 4, 256, 24, 1025), (128, 8, 1024, 16, 9), (272, 1, 256, 16, 9), (240, 1, 1024, 32, 9)])
def test_both_sides_of_the_fused_selection(device, width, heads, slots, reads, batch):
    """Routes selected in the prepare's launch and in their own (more than
    4,096 rows, or more than five rounds of a chunk of inputs in the fused
    kernel): the same bits, which are product_key_routes' of the keys."""

    from copy_on_write_sdm_amd import _native as nat
    from copy_on_write_sdm_amd.routing import product_key_routes

    print(f"fused selection width={width} H={heads} N={slots} R={reads} B={batch}", flush=True)
    layer = make_layer(width, slots=slots, reads=reads, writes=4, heads=heads, seed=batch,
                       dtype=torch.float32)
    c = ctl.SDMController.from_module(layer, device=device)
    x = torch.randn(batch, 1, width, device=device)
    inp = ctl.prepare_sdm_step(c, x).inputs
    rows, key = batch * heads, c.key_width_per_head
    f = lambda *shape: torch.empty(*shape, device=device)
    normalized, read_keys, write_keys = f(batch, width), f(rows, 1, key), f(rows, 1, key)
    values, gate, forget = f(rows, c.head_width), f(rows), f(rows)
    nat.check(nat.lib().cowsdm_controller_prepare(
        c.c_struct(), x.data_ptr(), batch, normalized.data_ptr(), read_keys.data_ptr(),
        write_keys.data_ptr(), values.data_ptr(), gate.data_ptr(), forget.data_ptr(),
        nat.stream_handle(device)), "prepare")
    assert torch.equal(inp.values, values) and torch.equal(inp.forget_log_gate, forget)
    for keys, k, name in ((read_keys, reads, "read"), (write_keys, 4, "write")):
        weights, indices = product_key_routes(keys, slots=slots, selected=k)
        assert torch.equal(getattr(inp, f"{name}_indices"), indices[:, 0])
        assert torch.equal(getattr(inp, f"{name}_weights"), weights[:, 0])
    alone = ctl.prepare_sdm_step(c, x[-1:]).inputs
    assert torch.equal(alone.read_indices, inp.read_indices[-heads:])
    assert torch.equal(alone.read_weights, inp.read_weights[-heads:])
