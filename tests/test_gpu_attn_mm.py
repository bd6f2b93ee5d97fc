"""Causal prefill attention on the matrix cores (lt_attn_mm.hip) at the sizes where it can go
wrong, against the oracle bit for bit: tiles of 16 query rows and of 16 positions with their
remainders, chunks of the positions held in LDS (512 and 1024) and one past them, few and many
tiles, cache values that are not finite in the rows that only part of a tile attends, query rows
at an odd stride, and splits whose lengths are not multiples of a V block, of up to 32 positions (a half-wave each in the
softmax), 33 and 34, 64 to 66 and 87 (a wave each, one and several V blocks)."""
import ctypes

import numpy as np
import pytest

from llamatov_amd import _lib
from llamatov_amd import engine as dr
from llamatov_amd._lib import LT_KV_F16, LT_KV_F32, call

pytestmark = pytest.mark.gpu


def _run(gpu, oracle, kv_dtype, nh, nkv, hd, len0, T, maxt, nsplit, rows, seed, odd_stride=0, bad=(), end=0):
    f16 = kv_dtype == LT_KV_F16
    print(f"[gpu-case] attn mm nh={nh} nkv={nkv} hd={hd} f16={f16} len0={len0} T={T} maxt={maxt} "
          f"nsplit={nsplit} bad={bad} end={end}", flush=True)
    rng = np.random.default_rng(seed)
    stride = nh * hd + odd_stride
    q = rng.standard_normal((T, stride)).astype(np.float32)
    k, v = (rng.standard_normal((maxt, nkv * hd)).astype(np.float32) for _ in range(2))
    if f16:
        k, v = k.astype(np.float16), v.astype(np.float16)
    k[len0 + T:], v[len0 + T:] = np.nan, np.nan
    for row, value in bad:
        v[row, :: 7] = value
    kd, vd = (a.view(np.uint16) if f16 else a for a in (k, v))
    up = lambda a: dr.DevTensor.from_host(a, gpu)
    ws_n = _lib.raw("lt_attn_workspace_size")(T, nh, hd, nsplit)
    ws = dr.DevTensor.empty((max(ws_n, 1),), np.uint8, gpu)
    out = dr.DevTensor.empty((T, nh * hd), np.float32, gpu)
    scale = float(hd ** -0.5)
    ts = [up(q), up(kd), up(vd), up(np.array([len0], np.int32))]
    call("lt_attn_prefill_end", gpu.handle, ts[0].vp, stride, ts[1].vp, ts[2].vp, ts[3].vp, out.vp, T, nh, nkv, hd,
         ctypes.c_float(scale), maxt, nsplit, kv_dtype, ws.vp, ws.nbytes, end)
    got = out.to_host()
    for t in rows:
        exp = oracle.attn_decode(np.ascontiguousarray(q[t, : nh * hd]), kd, vd, len0 + t + 1, nh, nkv, hd, scale, f16,
                                 nsplit)
        same = (got[t].view(np.uint32) == exp.view(np.uint32)) | (np.isnan(got[t]) & np.isnan(exp))
        assert same.all(), f"query {t} L={len0 + t + 1}: {np.flatnonzero(~same)[:5]}"
    for t in ts + [ws, out]:
        t.free()


@pytest.mark.parametrize("kv_dtype,nh,nkv,hd", [(LT_KV_F16, 14, 2, 64), (LT_KV_F32, 4, 4, 128),
                                                 (LT_KV_F16, 4, 2, 128), (LT_KV_F32, 3, 1, 64)])
@pytest.mark.parametrize("len0,T", [(0, 1), (0, 15), (0, 16), (0, 17), (3, 65), (31, 33), (49, 64)])
def test_tile_edges(gpu, oracle, kv_dtype, nh, nkv, hd, len0, T):
    _run(gpu, oracle, kv_dtype, nh, nkv, hd, len0, T, len0 + T + 3, 1, range(T), 5 * T + len0, odd_stride=3)


@pytest.mark.parametrize("kv_dtype", [LT_KV_F16, LT_KV_F32])
@pytest.mark.parametrize("nh,nkv,hd", [(14, 2, 64), (4, 1, 128)])
@pytest.mark.parametrize("len0,T", [(0, 32), (1, 32), (40, 24), (41, 24), (0, 112), (96, 17), (0, 200)])
@pytest.mark.parametrize("end", [0, None, 1, 1 << 30])
def test_context_end(gpu, oracle, kv_dtype, nh, nkv, hd, len0, T, end):
    """The known end of the context, at both sides of each line it draws, unknown and wrong."""
    rows = sorted({0, 1, 15, 16, T - 17, T - 1})
    _run(gpu, oracle, kv_dtype, nh, nkv, hd, len0, T, 400, 1, rows, T + len0, odd_stride=1,
         end=len0 + T if end is None else end)


# (few workgroups: 8 waves and chunks of 1024; more than one per CU: 4 waves and chunks of 512)
@pytest.mark.parametrize("kv_dtype,nh,hd,len0,T", [(LT_KV_F16, 2, 128, 1000, 40), (LT_KV_F32, 2, 64, 2030, 20),
                                                    (LT_KV_F16, 64, 64, 440, 140), (LT_KV_F32, 32, 128, 500, 144),
                                                    (LT_KV_F16, 32, 128, 1000, 144)])
def test_chunk_edges(gpu, oracle, kv_dtype, nh, hd, len0, T):
    rows = sorted({0, 1, 11, 12, 13, 23, 24, 25, T // 2, T - 1} & set(range(T)))
    _run(gpu, oracle, kv_dtype, nh, 1, hd, len0, T, len0 + T + 5, 1, rows, T + hd)


@pytest.mark.parametrize("kv_dtype", [LT_KV_F16, LT_KV_F32])
@pytest.mark.parametrize("hd,len0,T,nsplit", [(64, 5, 40, 1), (128, 0, 48, 1), (64, 0, 400, 16), (128, 0, 400, 32),
                                              (64, 300, 400, 16), (128, 700, 400, 16)])
def test_values_not_finite(gpu, oracle, kv_dtype, hd, len0, T, nsplit):
    """An infinity or a nan in the cache reaches exactly the queries that attend its row."""
    n = len0 + T
    _run(gpu, oracle, kv_dtype, 4, 2, hd, len0, T, n + 2, nsplit, range(max(0, T - 40), T), hd + T,
         bad=((n - 12, np.inf), (n - 5, np.nan), (n - 1, -np.inf)))


@pytest.mark.parametrize("kv_dtype,hd", [(LT_KV_F16, 64), (LT_KV_F32, 64), (LT_KV_F16, 128), (LT_KV_F32, 128)])
@pytest.mark.parametrize("len0,T,maxt,nsplit", [(0, 400, 512, 16), (7, 385, 700, 16), (0, 390, 400, 128),
                                                 (300, 384, 1500, 48), (0, 530, 700, 16), (627, 400, 1100, 16),
                                                 (640, 401, 1041, 16), (1000, 384, 1600, 16)])
def test_splits(gpu, oracle, kv_dtype, hd, len0, T, maxt, nsplit):
    rows = sorted({0, 1, 15, 16, 17, 100, 255, 256, 257, T - 18, T - 17, T - 2, T - 1})
    _run(gpu, oracle, kv_dtype, 4, 2, hd, len0, T, maxt, nsplit, rows, T + nsplit, odd_stride=1)
