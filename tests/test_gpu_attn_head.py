"""Unsplit decode attention with a workgroup per head (lt_attn_head.hip) at the lengths where it
can go wrong, against the oracle bit for bit: the 64-position score rounds and their spread over 8
waves (512 positions, 1024), the 16- and 32-row V blocks and the 256 rows in flight, both cache
types and head sizes, the step's new row at each of those places, nan past the length; batches of as
many (sequence, head) pairs as there are CUs and one more sequence; and past that a workgroup per KV
group (2 to 16 heads, tiles of 16 positions, 128 and 256 of them in flight) and the first groups
that it leaves to the general kernel (17 heads, more groups than CUs)."""
import ctypes

import numpy as np
import pytest

from llamatov_amd import engine as dr
from llamatov_amd._lib import LT_KV_F16, LT_KV_F32, call

pytestmark = pytest.mark.gpu

LENS = (1, 15, 16, 17, 31, 33, 64, 65, 255, 256, 257, 511, 513, 1024, 1025, 1290)
# exps one, two or four at a time; one position a thread or more
EXP_LENS = (63, 127, 128, 129, 192, 193, 320, 321, 384, 385, 449, 512)


def _cache(rng, shape, f16):
    x = rng.standard_normal(shape).astype(np.float32)
    return x.astype(np.float16).view(np.uint16) if f16 else x


@pytest.mark.parametrize("kv_dtype", [LT_KV_F32, LT_KV_F16])
@pytest.mark.parametrize("nh,nkv,hd", [(2, 1, 64), (3, 3, 128)])
def test_step_lengths(gpu, oracle, kv_dtype, nh, nkv, hd):
    _step(gpu, oracle, kv_dtype, nh, nkv, hd, LENS)


@pytest.mark.parametrize("kv_dtype", [LT_KV_F32, LT_KV_F16])
@pytest.mark.parametrize("nh,nkv,hd", [(2, 1, 64), (7, 7, 128)])
def test_step_exps(gpu, oracle, kv_dtype, nh, nkv, hd):
    _step(gpu, oracle, kv_dtype, nh, nkv, hd, EXP_LENS)


# (less LDS for the exps than threads: only the context's own are read)
@pytest.mark.parametrize("kv_dtype", [LT_KV_F32, LT_KV_F16])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("maxt", [1, 20, 256, 300])
def test_small_caches(gpu, oracle, kv_dtype, hd, maxt):
    _step(gpu, oracle, kv_dtype, 2, 1, hd, (1, min(maxt, 17)), maxt)
    _batched(gpu, oracle, kv_dtype, 2, 1, hd, 3, (1, maxt, min(maxt, 17)), maxt)


def _step(gpu, oracle, kv_dtype, nh, nkv, hd, lens, maxt=1300):
    f16, theta = kv_dtype == LT_KV_F16, 1e6
    rng = np.random.default_rng(hd)
    width, scale = nkv * hd, float(hd ** -0.5)
    up = lambda a: dr.DevTensor.from_host(a, gpu)
    freqs = up(oracle.rope_freqs(hd, theta))
    base_k, base_v = _cache(rng, (maxt, width), f16), _cache(rng, (maxt, width), f16)
    nan = 0x7E00 if f16 else np.nan
    for L in (0,) + tuple(n - 1 for n in lens[1:]) + (maxt - 1,):
        print(f"[gpu-case] attn head step nh={nh} hd={hd} f16={f16} L={L}", flush=True)
        kc, vc = base_k.copy(), base_v.copy()
        kc[L:], vc[L:] = nan, nan
        qkv = rng.standard_normal(nh * hd + 2 * width).astype(np.float32)
        roped = oracle.rope(qkv[: (nh + nkv) * hd], L, nh + nkv, hd, theta)
        ek, ev = kc.copy(), vc.copy()
        for dst, new in ((ek, roped[nh * hd:]), (ev, qkv[(nh + nkv) * hd:])):
            dst[L] = new.astype(np.float16).view(np.uint16) if f16 else new
        exp = oracle.attn_decode(roped[: nh * hd], ek, ev, L + 1, nh, nkv, hd, scale, f16, 1)
        ts = [up(qkv), up(kc), up(vc), up(np.array([L], np.int32)), dr.DevTensor.empty((nh * hd,), np.float32, gpu),
              dr.DevTensor.empty((nh * hd,), np.int8, gpu), dr.DevTensor.empty((nh * hd // 32,), np.uint16, gpu)]
        call("lt_attn_step", gpu.handle, ts[0].vp, freqs.vp, ts[1].vp, ts[2].vp, ts[3].vp, ts[4].vp, ts[5].vp, ts[6].vp,
             nh, nkv, hd, ctypes.c_float(scale), maxt, 1, kv_dtype, None, 0)
        assert np.array_equal(ts[4].to_host().view(np.uint32), exp.view(np.uint32)), L
        xq, xd = oracle.quant_q8(exp)
        assert np.array_equal(ts[5].to_host(), xq) and np.array_equal(ts[6].to_host(), xd), L
        assert ts[1].to_host().tobytes() == ek.tobytes() and ts[2].to_host().tobytes() == ev.tobytes(), L
        for t in ts:
            t.free()


@pytest.mark.parametrize("kv_dtype", [LT_KV_F32, LT_KV_F16])
@pytest.mark.parametrize("nh,nkv,hd,B", [(14, 2, 64, 16), (4, 1, 128, 16), (64, 8, 64, 4), (64, 8, 64, 5),
                                          (14, 2, 64, 20), (32, 2, 128, 10), (8, 4, 64, 40), (80, 80, 64, 4), (51, 3, 64, 6)])
def test_batched_lengths(gpu, oracle, kv_dtype, nh, nkv, hd, B):
    _batched(gpu, oracle, kv_dtype, nh, nkv, hd, B, LENS)


# (odd counts of KV groups, of (sequence, group) pairs and of both, per head and per group)
@pytest.mark.parametrize("kv_dtype", [LT_KV_F32, LT_KV_F16])
@pytest.mark.parametrize("nh,nkv,hd,B", [(6, 3, 64, 23), (7, 7, 128, 30), (1, 1, 64, 25), (32, 8, 128, 15), (21, 3, 64, 25)])
def test_batched_exps(gpu, oracle, kv_dtype, nh, nkv, hd, B):
    _batched(gpu, oracle, kv_dtype, nh, nkv, hd, B, EXP_LENS + (1, 2))


def _batched(gpu, oracle, kv_dtype, nh, nkv, hd, B, all_lens, maxt=1300):
    f16 = kv_dtype == LT_KV_F16
    rng = np.random.default_rng(B * hd)
    width, scale = nkv * hd, float(hd ** -0.5)
    up = lambda a: dr.DevTensor.from_host(a, gpu)
    lens = [all_lens[(5 * b + 3) % len(all_lens)] for b in range(B)]
    print(f"[gpu-case] attn head batch nh={nh} hd={hd} f16={f16} B={B} lens={lens}", flush=True)
    k, v = _cache(rng, (B, maxt, width), f16), _cache(rng, (B, maxt, width), f16)
    for b, L in enumerate(lens):
        k[b, L:], v[b, L:] = (0x7E00, 0x7E00) if f16 else (np.nan, np.nan)
    stride = nh * hd + 5
    q = rng.standard_normal((B, stride)).astype(np.float32)
    ts = [up(q), up(k), up(v), up(np.array(lens, np.int32)), dr.DevTensor.empty((B, nh * hd), np.float32, gpu),
          dr.DevTensor.empty((nh * hd // 32, B, 32), np.int8, gpu), dr.DevTensor.empty((nh * hd // 32, B), np.uint16, gpu)]
    call("lt_attn_decode_rows_q8_bm", gpu.handle, ts[0].vp, stride, ts[1].vp, ts[2].vp, ts[3].vp, ts[4].vp, ts[5].vp,
         ts[6].vp, B, nh, nkv, hd, ctypes.c_float(scale), maxt, kv_dtype)
    got, gq, gd = ts[4].to_host(), ts[5].to_host(), ts[6].to_host()
    for b, L in enumerate(lens):
        exp = oracle.attn_decode(np.ascontiguousarray(q[b, : nh * hd]), k[b], v[b], L, nh, nkv, hd, scale, f16, 1)
        assert np.array_equal(got[b].view(np.uint32), exp.view(np.uint32)), (b, L)
        xq, xd = oracle.quant_q8(exp)
        assert np.array_equal(gq[:, b].reshape(-1), xq) and np.array_equal(gd[:, b], xd), (b, L)
    for t in ts:
        t.free()
