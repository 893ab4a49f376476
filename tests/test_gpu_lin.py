"""The few-row matrix-core linear (vqk_lin.h) against the float64 oracle: every
x form, the edges of its row tiles, weight rows longer than one pass, ragged
last blocks, dead rows, and x that is not finite."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import vq_oracle as vo
from vq_cases import make_module, skipzero, to_device

pytestmark = pytest.mark.gpu

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _desc(m, row_table=None, sz=None):
    from vqlab_amd import _torch as Tt
    keep = []
    if sz is not None:
        st = np.ascontiguousarray(sz["sz_codes"])
        signed = {4: np.int32, 2: np.int16, 1: np.uint8}[st.itemsize]
        codes = torch.from_numpy(st.view(signed)).cuda()
        scales = torch.from_numpy(sz["sz_scales"]).cuda()
        cb = torch.from_numpy(m["codebook"]).cuda()
        rt = torch.from_numpy(row_table).cuda()
        return Tt.weights(codes, cb, scales, 64, m["pack_bits"], m["IN"], rt, keep=keep), keep
    codes, cb, sc = to_device(m)
    return Tt.weights(codes[0], cb, sc[0], 64, m["pack_bits"], m["IN"], keep=keep), keep


def _apply(w, x, scratch=True, fused=64, y_type=torch.float32):
    """vqk_linear_apply with the fused path up to `fused` rows."""
    from vqlab_amd import _lib as L, _torch as Tt
    N = x.shape[0]
    o = L.options(dense_fused_max_n=fused)
    ws = ctypes.c_size_t()
    L.check(L.lib().vqk_linear_apply_scratch(ctypes.byref(w), N, ctypes.byref(o), ctypes.byref(ws)))
    work = torch.full((max(1, ws.value),), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.full((N, w.OUT), float("nan"), dtype=y_type, device="cuda")
    L.check(L.lib().vqk_linear_apply(ctypes.byref(w), Tt.ptr(x), Tt.act_type(x), N, Tt.ptr(y),
                                     Tt.act_type(y), Tt.ptr(work) if scratch else None,
                                     ws.value if scratch else 0, ctypes.byref(o), Tt.stream()))
    torch.cuda.synchronize()
    return y.double().cpu().numpy()


def _weight(m, decoded):
    """float64 [OUT, IN]: the fp16 weight that the dequant writes, or (decoded
    False) the unrounded product of entry and scale."""
    if decoded:
        return vo.dequant(m["codes"][0], m["codebook"], m["scales"][0], 64).astype(np.float64)
    w = m["codebook"].astype(np.float64)[m["codes"][0]].reshape(m["OUT"], m["IN"])
    return w * np.repeat(m["scales"][0].astype(np.float64), 64, axis=1)


def _ref(m, x, rounded, decoded=False):
    """float64 product of x, or x rounded to fp16, with the module's weight;
    and the bar of fp32 accumulation: each of the n products and sums of a row,
    and the scaling of its groups' sums, rounds once, so n * 2^-24 of sum |w x|
    bounds the error of any order (n / 64 scalings, well under the n sums)."""
    w = _weight(m, decoded)
    xv = x.half() if rounded else x
    xv = xv.double().cpu().numpy()
    return xv @ w.T, np.abs(xv) @ np.abs(w).T * (m["IN"] * 2.0 ** -24)


# (d, K, packed, OUT, IN): more blocks per row than a GEMV wave holds or ragged
# last blocks, which this kernel takes at every size; OUT off the 16-row tile; a
# table in LDS, partly in LDS, and not in LDS at all
SHAPES = [
    (2, 256, False, 100, 4160), (2, 1024, True, 33, 4224), (4, 256, False, 40, 1344),
    (4, 4096, True, 130, 8448), (4, 8192, True, 17, 1088), (4, 65536, False, 48, 2112),
    (8, 4096, True, 65, 1088), (8, 16384, True, 40, 4160), (8, 65536, False, 33, 16640),
]


@pytest.mark.parametrize("d,K,packed,OUT,IN", SHAPES)
@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
def test_linear_rows(d, K, packed, OUT, IN, dt):
    rng = np.random.default_rng(d * 131 + K + IN)
    m = make_module(rng, 1, OUT, IN, d, K, packed=packed)
    w, keep = _desc(m)
    for N in (1, 2, 4, 5, 16, 17, 32, 33, 64):
        print(f"linear rows d{d} K{K} {IN}->{OUT} {dt} N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda().to(DT[dt])
        ref, bar = _ref(m, x, rounded=d != 8 or dt == "f16")
        y = _apply(w, x)
        assert (np.abs(y - ref) <= bar).all(), (N, np.abs(y - ref).max(), bar.min())


@pytest.mark.parametrize("d,bits", [(2, b) for b in range(8, 13)] +
                         [(d, b) for d in (4, 8) for b in (8, 9, 10, 11, 12, 13, 14, 16)])
def test_linear_rows_every_width(d, bits):
    """Every code width: whole supersteps and a ragged one, x in place and (past
    2^28 products) in operand order, the scale in fp32 and the decoded weight."""
    rng = np.random.default_rng(10 * d + bits)
    for OUT, IN, rows in ((33, 128 * d * 9 + 64, (3, 17)), (13201, 4160, (20, 40))):
        m = make_module(rng, 1, OUT, IN, d, 2 ** bits)
        w, keep = _desc(m)
        cols = np.arange(OUT) if OUT < 100 else rng.choice(OUT, 60, replace=False)
        sub = dict(m, codes=m["codes"][:, cols], scales=m["scales"][:, cols], OUT=len(cols))
        for N in rows:
            print(f"linear width d{d} bits {bits} {IN}->{OUT} N{N}", flush=True)
            x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda().half()
            for fused in (64, 0):
                ref, bar = _ref(sub, x, rounded=True, decoded=fused == 0)
                y = _apply(w, x, fused=fused)[:, cols]
                assert (np.abs(y - ref) <= bar).all(), (N, fused, np.abs(y - ref).max())


@pytest.mark.parametrize("d,K,packed,IN", [
    (2, 1024, True, 4160), (2, 256, False, 4096), (4, 4096, True, 4160), (4, 1024, True, 4096),
    (4, 65536, False, 4096), (8, 16384, True, 4160), (8, 4096, True, 4096), (8, 65536, False, 4160)])
def test_linear_rows_operand_order(d, K, packed, IN):
    """Shapes whose x is copied into operand order (2^28 products and more), with
    a ragged last block or whole supersteps, an odd OUT and dead rows, at the
    edges of the row tiles, against the oracle on sampled columns -- as without
    scratch, where x is read in place; an infinite and a NaN value of x stay in
    their rows."""
    from vqlab_amd import _lib as L
    rng = np.random.default_rng(d + K)
    m = make_module(rng, 1, 13201, IN, d, K, packed=packed, dead_frac=0.02)
    sz, rt = skipzero(m)
    w, keep = _desc(m, rt, sz)
    cols = np.unique(np.concatenate([rng.choice(m["OUT"], 150, replace=False), [0, 15, 16, 13199, 13200]]))
    sub = dict(m, codes=m["codes"][:, cols], scales=m["scales"][:, cols], OUT=len(cols))
    for N in (5, 16, 17, 32, 33, 49, 64):
        print(f"linear operand order d{d} K{K} {IN} N{N}", flush=True)
        o, ws = L.options(dense_fused_max_n=64), ctypes.c_size_t()
        L.check(L.lib().vqk_linear_apply_scratch(ctypes.byref(w), N, ctypes.byref(o), ctypes.byref(ws)))
        assert ws.value > 0
        x = torch.from_numpy(rng.standard_normal((N, m["IN"])).astype(np.float32)).cuda().half()
        for fused in (64, 0):                       # scales in fp32, and the decoded weight
            if fused == 0 and N <= 32:
                continue
            ref, bar = _ref(sub, x, rounded=True, decoded=fused == 0)
            for scratch in (True, False):
                if fused == 0 and not scratch and m["IN"] % (32 * d):
                    continue                        # the ragged dense GEMM's own workspace
                y = _apply(w, x, scratch, fused)[:, cols]
                assert (np.abs(y - ref) <= bar).all(), (N, fused, scratch, np.abs(y - ref).max(), bar.min())
                assert not np.signbit(y[:, rt[0][cols] < 0]).any()
        y = _apply(w, x)[:, cols]
        if d != 8:                                  # bf16 / fp32 rounded on the way
            assert np.array_equal(_apply(w, x.float())[:, cols], y)
        x[1, 7], x[3, IN - 1] = float("inf"), float("nan")
        y = _apply(w, x)
        live = rt[0] >= 0
        assert np.isfinite(y[[0, 2] + list(range(4, N))]).all()
        assert not np.isfinite(y[1][live]).any() and np.isnan(y[3][live]).all()


@pytest.mark.parametrize("d,K,packed", [(2, 1024, True), (4, 4096, True), (8, 4096, True),
                                        (8, 65536, False)])
def test_linear_rows_scale_in_fp32(d, K, packed):
    """The scale multiplies a group's fp32 sum, not the fp16 entry: products of
    entry and scale above fp16's range (rows 0, 3, ...) and among its subnormals
    (rows 1, 4, ...) come out as exactly as the others, whatever the row count;
    IN leaves the last superstep one block, or one and half a block."""
    rng = np.random.default_rng(d + K)
    IN = 64 * 65 if d == 2 else 64 * 33         # no fast GEMV: more than 64 blocks, or a ragged one
    m = make_module(rng, 1, 50, IN, d, K, packed=packed, cb_std=2.0)
    m["scales"][0, 0::3] *= np.float16(40000)
    m["scales"][0, 1::3] *= np.float16(2.0 ** -12)
    m["codebook"][: K // 2] *= np.float16(2.0 ** -10)
    w, keep = _desc(m)
    prod = np.abs(_weight(m, False))
    assert prod.max() > 65504 and (prod[1::3] < 2.0 ** -14).mean() > 0.5
    for dt in DT:
        for N in (2, 7, 16, 20, 32):
            print(f"linear scale d{d} K{K} {dt} N{N}", flush=True)
            x = torch.from_numpy(rng.standard_normal((N, m["IN"])).astype(np.float32)).cuda().to(DT[dt])
            ref, bar = _ref(m, x, rounded=d != 8 or dt == "f16")
            y = _apply(w, x)
            assert (np.abs(y - ref) <= bar).all(), (N, np.abs(y - ref).max(), bar.min())


# (d, K, packed, OUT, IN, x, rows): both sides of each size from which the few-row
# kernel takes over from the GEMV (20, 40, 70, 30, 90 and 40 million products)
EDGES = [(2, 256, False, 1024, 2048, "f16", (9, 10)), (4, 4096, True, 1024, 4096, "bf16", (9, 10)),
         (8, 4096, True, 2048, 2048, "f16", (16, 17)), (8, 16384, True, 1024, 2048, "f16", (14, 15)),
         (8, 4096, True, 1024, 4096, "bf16", (2, 21, 22)), (8, 65536, False, 1024, 2048, "f32", (19, 20))]


@pytest.mark.parametrize("d,K,packed,OUT,IN,dt,rows", EDGES)
def test_linear_rows_at_the_gemv_edge(d, K, packed, OUT, IN, dt, rows):
    """Rows on both sides of the size from which the few-row kernel runs in
    place of the GEMV: one arithmetic, the same bar."""
    rng = np.random.default_rng(d + K)
    m = make_module(rng, 1, OUT, IN, d, K, packed=packed)
    w, keep = _desc(m)
    for N in rows:
        print(f"linear edge d{d} K{K} {dt} N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda().to(DT[dt])
        ref, bar = _ref(m, x, rounded=d != 8 or dt == "f16")
        assert (np.abs(_apply(w, x) - ref) <= bar).all(), N


# both sides of each line between the segment kernel and the few-row kernel
SEG_EDGES = [(2, 1024, True, 6400, 1024, (48, 49)), (4, 4096, True, 256, 1024, (40,)), (4, 4096, True, 256, 1536, (40,)),
             (4, 1024, True, 8576, 2048, (33, 48, 49)), (4, 8192, True, 8576, 1536, (48, 49)), (4, 8192, True, 8192, 1024, (48, 64)),
             (8, 4096, True, 16384, 3072, (16, 17, 33)), (8, 4096, True, 256, 2048, (8, 40)),
             (8, 16384, True, 256, 2048, (32, 33)), (8, 65536, False, 8192, 1024, (48, 64))]


@pytest.mark.parametrize("d,K,packed,OUT,IN,rows", SEG_EDGES)
def test_linear_rows_at_the_segment_edge(d, K, packed, OUT, IN, rows):
    """The same for the decoded-weight path (every row through vqk_dense_gemm):
    the oracle on sampled columns, x rounded to fp16, W the dequant's fp16."""
    rng = np.random.default_rng(d + K)
    m = make_module(rng, 1, OUT, IN, d, K, packed=packed)
    w, keep = _desc(m)
    cols = rng.choice(OUT, min(OUT, 300), replace=False)
    sub = dict(m, codes=m["codes"][:, cols], scales=m["scales"][:, cols], OUT=len(cols))
    for N in rows:
        print(f"linear segment edge d{d} K{K} {IN}->{OUT} N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda()
        ref, bar = _ref(sub, x, rounded=True, decoded=True)
        assert (np.abs(_apply(w, x, fused=0)[:, cols] - ref) <= bar).all(), N


def test_linear_rows_keep_x():
    """d8 takes bf16 / fp32 x unrounded: values below fp16's smallest and above
    its largest come through."""
    rng = np.random.default_rng(5)
    m = make_module(rng, 1, 48, 2112, 8, 4096)
    w, keep = _desc(m)
    for dt in ("bf16", "f32"):
        print(f"linear keeps x {dt}", flush=True)
        x = torch.from_numpy(rng.standard_normal((3, m["IN"])).astype(np.float32)).cuda()
        x[1] *= 2.0 ** -30
        x[2] *= 2.0 ** 20
        x = x.to(DT[dt])
        ref, bar = _ref(m, x, rounded=False)
        assert (np.abs(_apply(w, x) - ref) <= bar).all()


@pytest.mark.parametrize("d,K,IN", [(4, 4096, 1088), (8, 16384, 1088), (2, 1024, 4224)])
def test_linear_rows_not_finite(d, K, IN):
    """An infinite or NaN value of one row of x stays in that row, also where
    the row's end is inside a block (its neighbour's values follow in memory)."""
    rng = np.random.default_rng(7 + d)
    m = make_module(rng, 1, 40, IN, d, K)
    w, keep = _desc(m)
    for N in (3, 9, 40):
        print(f"linear not finite d{d} N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda()
        x[1, 0], x[2, 3] = float("inf"), float("nan")
        y = _apply(w, x.half())
        assert np.isfinite(y[[0] + list(range(3, N))]).all()
        w0 = vo.dequant(m["codes"][0], m["codebook"], m["scales"][0], 64)[:, 0]
        assert np.array_equal(y[1][w0 != 0], np.sign(w0[w0 != 0]) * np.inf) and np.isnan(y[2]).all()


def test_linear_rows_dead():
    """Dead skipzero rows are +0, the live ones as in the expanded module."""
    rng = np.random.default_rng(11)
    m = make_module(rng, 1, 70, 1088, 4, 4096, dead_frac=0.3)
    sz, rt = skipzero(m)
    w, keep = _desc(m, rt, sz)
    full, keep2 = _desc(m)
    for N in (3, 20, 40):
        print(f"linear dead rows N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, m["IN"])).astype(np.float32)).cuda().half()
        y, ref = _apply(w, x), _apply(full, x)
        assert np.array_equal(y, ref) and not np.signbit(y[:, rt[0] < 0]).any()


@pytest.mark.parametrize("d,K,packed,IN", [(4, 4096, True, 1088), (4, 256, False, 4160), (8, 4096, True, 1088),
                                           (8, 65536, False, 4160)])
def test_linear_ragged_past_fused_rows(d, K, packed, IN):
    """33..64 rows of weight rows with a ragged last block at the default
    options multiply in x's own arithmetic: fp32 x to 16 significant bits (two
    bf16 parts: 2^-17 of each term, beside the fp32 sums), bf16 x beyond fp16's
    range finite, against W rounded once to bf16; fp16 x against the decoded
    weight."""
    rng = np.random.default_rng(d + IN)
    m = make_module(rng, 1, 70, IN, d, K, packed=packed)
    w, keep = _desc(m)
    for N in (33, 48, 64):
        print(f"linear ragged d{d} K{K} {IN} N{N}", flush=True)
        x = torch.from_numpy(rng.standard_normal((N, IN)).astype(np.float32)).cuda()
        ref, bar = _ref(m, x, rounded=False, decoded=True)
        bar = bar + bar / (IN * 2.0 ** -24) * 2.0 ** -17
        assert (np.abs(_apply(w, x, fused=32) - ref) <= bar).all()
        ref, bar = _ref(m, x, rounded=True, decoded=True)
        assert (np.abs(_apply(w, x.half(), fused=32) - ref) <= bar).all()
        big = (x * 1e6).bfloat16()
        wb = vo.bf16_values(_weight(m, True).astype(np.float32)).astype(np.float64)
        xb = big.double().cpu().numpy()
        y = _apply(w, big, fused=32)
        assert (np.abs(y - xb @ wb.T) <= np.abs(xb) @ np.abs(wb).T * (IN * 2.0 ** -24)).all()
