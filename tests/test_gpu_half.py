"""The half-entry segment kernel (vqk_half.h: d8 tables of 256 KB) through the
MoE block against the oracle: one and several 32-row tiles an expert, odd block
counts, row blocks with idle waves, dead rows, a shared expert,
every x type; and a workspace that has no room for its half sums."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from test_gpu_wide import _block, _oracle, _spec
from vq_cases import PATH_GROUPED, assert_close, moe_path

pytestmark = pytest.mark.gpu

CASES = [
    # E, H, I, K, k, T, shared, dead
    (8, 512, 256, 16384, 2, 100, False, 0.0),
    (4, 768, 256, 16384, 2, 190, True, 0.2),
    (3, 256, 768, 16384, 2, 70, False, 0.0),
    (64, 1280, 512, 16384, 4, 16, True, 0.0),
    (96, 512, 1280, 16384, 3, 70, True, 0.3),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_moe_half_entries(case, dt):
    E, H, I, K, k, T, shared, dead = case
    print(f"moe half entries {case} {dt}", flush=True)
    rng = np.random.default_rng(sum(case[:6]))
    blk, ms, sh, vec = _block(rng, E, H, I, 8, K, k, shared, dead)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).cuda().to(dt)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[: T // 2, 0] += 3.0                       # expert 0 gets more than one tile
    assert moe_path(blk, T) == PATH_GROUPED
    y = blk(x, torch.from_numpy(logits).cuda())
    assert torch.equal(y, blk(x, torch.from_numpy(logits).cuda()))
    kw = {}
    if shared:
        kw = dict(shared_gate=_spec(sh["gate"]), shared_up=_spec(sh["up"]), shared_down=_spec(sh["down"]),
                  shared_gate_vec=vec)
    assert_close(y.float().cpu().numpy(), _oracle(x, logits, ms, k, kw), what=f"moe half entries {case}")


def test_moe_half_entries_not_finite():
    """A token with an infinite activation changes no other token's row."""
    print("moe half entries not finite", flush=True)
    rng = np.random.default_rng(3)
    blk, _, _, _ = _block(rng, 4, 768, 256, 8, 16384, 2)
    T = 150
    x = torch.from_numpy(rng.standard_normal((T, 768)).astype(np.float32)).cuda().half()
    lg = torch.from_numpy(rng.standard_normal((T, 4)).astype(np.float32)).cuda()
    y = blk(x, lg)
    x[7, 0] = float("inf")
    z = blk(x, lg)
    keep = [i for i in range(T) if i != 7]
    assert torch.equal(z[keep], y[keep]) and not torch.isfinite(z[7]).any()


def test_moe_half_entries_workspace():
    """A workspace with room for the 16-row kernel's rows only still runs the
    call (on that kernel); the full one gives the same within the oracle's bar."""
    from vqlab_amd import _lib as L, _torch as Tt
    print("moe half entries workspace", flush=True)
    rng = np.random.default_rng(11)
    E, H, I, k, T = 8, 512, 256, 2, 100
    blk, ms, _, _ = _block(rng, E, H, I, 8, 16384, k)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).cuda().half()
    logits = rng.standard_normal((T, E)).astype(np.float32)
    lg = torch.from_numpy(logits).cuda()
    ref = _oracle(x, logits, ms, k, {})
    keep, need = [], ctypes.c_size_t()
    d = blk._fused_desc(keep)
    L.check(L.lib().vqk_moe_decode_layer_workspace(ctypes.byref(d), T, ctypes.byref(need)))
    for size in (need.value, need.value - 256):
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
        y = torch.empty_like(x)
        L.check(L.lib().vqk_moe_decode_layer(ctypes.byref(d), Tt.ptr(x), L.VQK_F16, T, Tt.ptr(lg), Tt.ptr(y),
                                             L.VQK_F16, None, None, Tt.ptr(ws), size, Tt.stream()))
        assert_close(y.float().cpu().numpy(), ref, what=f"workspace of {size}")
