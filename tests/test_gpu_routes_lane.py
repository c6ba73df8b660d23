"""The lane-per-row route selection (csrc/routes.h) at the edges of its
networks: against oracle/routes.py (indices exactly, weights within rtol
2e-6 / atol 1e-7 as in test_gpu_routes.py), and against the wave-per-row
selection, which fewer rows take, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import copy_on_write_sdm_amd as cow
from oracle import routes

pytestmark = pytest.mark.gpu

LANE_ROWS = 4096   # rows from which sqrt(N) <= 32 is selected lane by lane, K = 9 .. 16 from
                   # twice as many


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("root,selected", [
    (1, 1), (2, 3), (5, 4), (9, 8), (16, 4), (16, 16), (15, 9), (16, 17), (7, 32),
    (17, 4), (32, 8), (31, 16), (32, 32), (20, 31)])
def test_lane_rows_equal_oracle_and_wave_rows(device, root, selected, ties):
    print(f"lane routes root={root} k={selected} ties={ties}", flush=True)
    rows, slots = LANE_ROWS + 37, root * root
    selected = min(selected, slots)
    rng = np.random.default_rng(root * 100 + selected)
    p = (rng.integers(-1, 2, size=(rows, 1, 2 * root)) * -0.5 if ties
         else rng.standard_normal((rows, 1, 2 * root))).astype(np.float32)
    x = torch.from_numpy(p).to(device)
    w, i = cow.product_key_routes(x, slots=slots, selected=selected)
    ew, ei = routes.product_key_routes(p[:300], slots, selected)
    np.testing.assert_array_equal(i[:300].cpu().numpy(), ei)
    np.testing.assert_allclose(w[:300].cpu().numpy(), ew, rtol=2e-6, atol=1e-7)
    # one more float of offset: unaligned rows take the general lane form, and
    # 2,000 rows at a time the wave form
    shifted = torch.empty(x.numel() + 1, device=device)[1:].view_as(x).copy_(x)
    parts = [cow.product_key_routes(shifted[a:a + 2000], slots=slots, selected=selected)
             for a in range(0, rows, 2000)]
    assert torch.equal(i, torch.cat([part[1] for part in parts]))
    assert torch.equal(w, torch.cat([part[0] for part in parts]))
    w2, i2 = cow.product_key_routes(shifted, slots=slots, selected=selected)
    assert torch.equal(i, i2) and torch.equal(w, w2)


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("root,selected", [
    (16, 16), (15, 9), (16, 9), (9, 12), (31, 16), (32, 16), (20, 13), (32, 9)])
def test_lane_rows_of_nine_to_sixteen_routes(device, root, selected, ties):
    """The form of both large prefills (N = 256, K = 16): from 8,192 rows, in
    the filled network and the general one, against the oracle and against
    2,000 rows at a time (sorted across lanes), bit for bit."""

    print(f"lane routes root={root} k={selected} ties={ties}", flush=True)
    rows, slots = 2 * LANE_ROWS + 37, root * root
    rng = np.random.default_rng(root * 100 + selected)
    p = (rng.integers(-1, 2, size=(rows, 1, 2 * root)) * -0.5 if ties
         else rng.standard_normal((rows, 1, 2 * root))).astype(np.float32)
    x = torch.from_numpy(p).to(device)
    w, i = cow.product_key_routes(x, slots=slots, selected=selected)
    some = np.r_[0:200, rows - 100:rows]
    ew, ei = routes.product_key_routes(p[some], slots, selected)
    np.testing.assert_array_equal(i.cpu().numpy()[some], ei)
    np.testing.assert_allclose(w.cpu().numpy()[some], ew, rtol=2e-6, atol=1e-7)
    parts = [cow.product_key_routes(x[a:a + 2000], slots=slots, selected=selected)
             for a in range(0, rows, 2000)]
    shifted = torch.empty(x.numel() + 1, device=device)[1:].view_as(x).copy_(x)
    w2, i2 = cow.product_key_routes(shifted, slots=slots, selected=selected)
    for got_w, got_i in ((torch.cat([part[0] for part in parts]),
                          torch.cat([part[1] for part in parts])), (w2, i2)):
        assert torch.equal(i, got_i) and torch.equal(w, got_w)
