"""The many-rows segment kernel (vqk_wide.h) through the MoE block against the
oracle: tile edges (32 / 64 / 96 rows and more than one tile an expert), odd
block counts, dead rows, a shared expert, every x type, and the sort's limits."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import vq_oracle as vo
from vq_cases import PATH_GROUPED, assert_close, make_module, moe_path, skipzero, to_device

pytestmark = pytest.mark.gpu


def _lin(m, sz):
    from vqlab_amd.vq_switch import VQSwitchLinear
    if not sz:
        codes, cb, sc = to_device(m)
        return VQSwitchLinear(codes, cb, sc, pack_bits=m["pack_bits"], in_features=m["IN"])
    c, rt = skipzero(m)
    return VQSwitchLinear(torch.from_numpy(np.ascontiguousarray(c["sz_codes"]).view(np.int32)).cuda(),
                          torch.from_numpy(m["codebook"]).cuda(), torch.from_numpy(c["sz_scales"]).cuda(),
                          pack_bits=m["pack_bits"], in_features=m["IN"], row_table=torch.from_numpy(rt).cuda())


def _spec(m):
    return {"codes": m["codes"], "codebook": m["codebook"], "scales": m["scales"], "group": 64}


def _block(rng, E, H, I, d, K, k, shared=False, dead=0.0):
    from vqlab_amd.moe import VQSparseMoeBlock, VQSwitchGLU
    dims = {"gate": (I, H), "up": (I, H), "down": (H, I)}
    ms = {n: make_module(rng, E, o, i, d, K, dead_frac=dead) for n, (o, i) in dims.items()}
    sh = {n: make_module(rng, 1, o, i, d, K) for n, (o, i) in dims.items()} if shared else None
    vec = (rng.standard_normal(H) / np.sqrt(H)).astype(np.float32) if shared else None
    glu = VQSwitchGLU(*(_lin(ms[n], dead > 0) for n in ("gate", "up", "down")))
    shg = VQSwitchGLU(*(_lin(sh[n], False) for n in ("gate", "up", "down"))) if shared else None
    blk = VQSparseMoeBlock(glu, k, True, shg, torch.from_numpy(vec).cuda() if shared else None)
    return blk, ms, sh, vec


CASES = [
    # E, H, I, d, K, k, T, shared, dead: pairs per expert in tiles of 1, 2 and 3
    # times 32 rows and over; odd block counts at d8 (H 768: 3, I 256: 1); two
    # tables of 64 KB (64-row tiles); many small experts
    (8, 512, 256, 4, 4096, 2, 100, False, 0.0),
    (4, 512, 384, 4, 1024, 2, 190, True, 0.0),
    (4, 768, 256, 8, 4096, 2, 230, True, 0.2),
    (8, 256, 512, 8, 1024, 2, 64, False, 0.0),
    (3, 512, 256, 4, 8192, 2, 200, False, 0.3),
    (160, 256, 256, 8, 2048, 4, 80, False, 0.0),
    # the shared expert as wide tiles too (512 rows and more)
    (4, 512, 384, 4, 1024, 2, 520, True, 0.0),
    (4, 768, 256, 8, 4096, 2, 530, True, 0.2),
    # both sides of the pairs per expert from which wide tiles run: three over a
    # small table beside a shared expert, ten beside it over few experts and
    # where few workgroups walk a long row (four over a 64 KB table)
    (128, 256, 256, 4, 256, 2, 191, True, 0.0),
    (128, 256, 256, 4, 256, 2, 192, True, 0.0),
    (16, 256, 256, 4, 1024, 2, 79, True, 0.0),
    (16, 256, 256, 4, 1024, 2, 80, True, 0.0),
    (32, 2304, 256, 4, 8192, 2, 63, False, 0.2),
    (32, 2304, 256, 4, 8192, 2, 64, False, 0.2),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_moe_many_rows(case, dt):
    E, H, I, d, K, k, T, shared, dead = case
    print(f"moe many rows {case} {dt}", flush=True)
    rng = np.random.default_rng(sum(case[:7]))
    blk, ms, sh, vec = _block(rng, E, H, I, d, K, k, shared, dead)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).cuda().to(dt)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[: T // 2, 0] += 3.0                       # expert 0 gets more than one tile
    assert moe_path(blk, T) == PATH_GROUPED
    y = blk(x, torch.from_numpy(logits).cuda())
    y2 = blk(x, torch.from_numpy(logits).cuda())
    assert torch.equal(y, y2)                        # tiles and sums do not depend on the pair order
    kw = {}
    if shared:
        kw = dict(shared_gate=_spec(sh["gate"]), shared_up=_spec(sh["up"]), shared_down=_spec(sh["down"]),
                  shared_gate_vec=vec)
    ref = _oracle(x, logits, ms, k, kw)
    assert_close(y.float().cpu().numpy(), ref, what=f"moe many rows {case}")


# E, H, I, d, K, k, T, shared, dead: enough experts that a workgroup walks several
# 256-row blocks of its tile -- two of three (H 768) and four of nine (H 2304) in
# down, the last workgroup fewer; two of three in gate and up (I 768)
BLOCK_CASES = [
    (256, 768, 128, 4, 1024, 2, 280, False, 0.0),
    (256, 2304, 128, 4, 4096, 2, 280, False, 0.2),
    (256, 768, 256, 8, 2048, 2, 200, True, 0.2),
    (256, 256, 768, 8, 1024, 2, 150, False, 0.2),
    (256, 512, 768, 4, 8192, 2, 260, False, 0.0),
]


@pytest.mark.parametrize("case", BLOCK_CASES)
def test_moe_several_row_blocks(case):
    """The walk over row blocks: the next block's rows and words taken up during
    the last superstep, x copies that wrap to its first chunk, stores between
    counted waits; dead rows and odd block counts (d8: 3 and 1) across it."""
    E, H, I, d, K, k, T, shared, dead = case
    blocks = -(-max(H, I) // 256)
    assert E * -(-blocks // 2) >= 512               # the grid rule's first step
    print(f"moe row blocks {case}", flush=True)
    rng = np.random.default_rng(sum(case[:7]))
    blk, ms, sh, vec = _block(rng, E, H, I, d, K, k, shared, dead)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).cuda().bfloat16()
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 3] += 2.0                              # expert 3 gets a tile of many rows
    assert moe_path(blk, T) == PATH_GROUPED
    y = blk(x, torch.from_numpy(logits).cuda())
    assert torch.equal(y, blk(x, torch.from_numpy(logits).cuda()))
    kw = {}
    if shared:
        kw = dict(shared_gate=_spec(sh["gate"]), shared_up=_spec(sh["up"]), shared_down=_spec(sh["down"]),
                  shared_gate_vec=vec)
    assert_close(y.float().cpu().numpy(), _oracle(x, logits, ms, k, kw), what=f"moe row blocks {case}")


def _oracle(x, logits, ms, k, kw):
    """vo.moe_layer of the routed experts plus the shared expert's term."""
    xf = x.float().cpu().numpy()
    ref, _, _ = vo.moe_layer(xf, logits, _spec(ms["gate"]), _spec(ms["up"]), _spec(ms["down"]), k,
                             h_round=np.float16)
    if kw:
        zero = np.zeros((xf.shape[0], 1), np.float32)
        one, _, _ = vo.moe_layer(xf, zero, kw["shared_gate"], kw["shared_up"], kw["shared_down"], 1,
                                 h_round=np.float16)
        g = 1.0 / (1.0 + np.exp(-(xf.astype(np.float64) @ kw["shared_gate_vec"].astype(np.float64))))
        ref = ref + g[:, None] * one
    return ref


def test_moe_many_rows_not_finite():
    """A token with an infinite activation changes no other token's row, with
    a block count (3) that leaves half of the last superstep without a block."""
    print("moe many rows not finite", flush=True)
    rng = np.random.default_rng(3)
    blk, ms, _, _ = _block(rng, 4, 768, 256, 8, 1024, 2)
    T = 150
    x = torch.from_numpy(rng.standard_normal((T, 768)).astype(np.float32)).cuda().half()
    lg = torch.from_numpy(rng.standard_normal((T, 4)).astype(np.float32)).cuda()
    y = blk(x, lg)
    x[7, 0] = float("inf")
    z = blk(x, lg)
    keep = [i for i in range(T) if i != 7]
    assert torch.equal(z[keep], y[keep]) and not torch.isfinite(z[7]).any()


@pytest.mark.parametrize("d,K", [(4, 1024), (8, 1024), (8, 16384)])
def test_moe_weight_beyond_fp16(d, K):
    """A weight that overflows fp16 (row 5 of every expert's down projection, one
    column) makes its output infinite, with the sign of what it multiplies, and
    changes no other; with an odd block count, whose last superstep has a lane
    group without a block (d8 16384: the half-entry kernel, same rule)."""
    print(f"moe weight beyond fp16 d{d} K{K}", flush=True)
    rng = np.random.default_rng(d)
    E, H, I, k, T = 4, 512, 32 * d * (1 if d == 8 else 3), 2, 100
    blk, ms, _, _ = _block(rng, E, H, I, d, K, k)
    m = ms["down"]
    m["codebook"][0] = 0
    m["codebook"][0, 0] = 2.0
    m["codes"][:, 5, -I // d:] = np.maximum(m["codes"][:, 5, -I // d:], 1)
    m["codes"][:, 5, -1] = 0
    m["scales"][:, 5, -1] = 60000.0
    m["stored"] = vo.pack(m["codes"], m["pack_bits"])
    blk.switch_mlp.down_proj = _lin(m, False)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).cuda().half()
    logits = rng.standard_normal((T, E)).astype(np.float32)
    y = blk(x, torch.from_numpy(logits).cuda()).double().cpu().numpy()
    with np.errstate(all="ignore"):
        ref = _oracle(x, logits, ms, k, {})
    same = ~np.isnan(ref[:, 5])                     # both experts' terms of one sign
    assert np.isinf(ref[same, 5]).all() and same.mean() > 0.3
    assert np.array_equal(y[same, 5], ref[same, 5]) and np.isnan(y[~same, 5]).all()
    rest = [r for r in range(H) if r != 5]
    assert_close(y[:, rest], ref[:, rest], what="beside a weight beyond fp16")


@pytest.mark.parametrize("N", [24 * 1024, 24 * 1024 + 8])
def test_sort_past_its_lds(N):
    """The pair order staged in LDS at its limit, and in place past it."""
    from vqlab_amd import vq_switch as VS
    print(f"sort {N}", flush=True)
    rng = np.random.default_rng(N)
    E, OUT, IN, k = 16, 16, 128, 8
    m = make_module(rng, E, OUT, IN, 4, 256, packed=False)
    codes, cb, sc = to_device(m)
    x = torch.from_numpy(rng.standard_normal((N // k, IN)).astype(np.float32)).cuda().half()
    ids = rng.integers(0, E, N).astype(np.int32)
    y = VS._gemmseg(x, torch.from_numpy(ids).cuda(), codes, cb, sc, 0, IN, k, out_dtype=torch.float32)
    w = vo.dequant(m["codes"].reshape(E * OUT, -1), m["codebook"], m["scales"].reshape(E * OUT, -1), 64)
    w = w.reshape(E, OUT, IN).astype(np.float64)
    xf = np.repeat(x.double().cpu().numpy(), k, axis=0)
    ref = np.einsum("ni,noi->no", xf, w[ids])
    assert_close(y.cpu().numpy(), ref, rtol=1e-4, atol=1e-4, what="sort")
