"""The tiled GEMM's choice of kernel (take_ls and gemm_walk in lt_prefill.hip): what it is at both sides of each
line of the rule, and that there the default launch gives the bits of k_q8_gemm's dynamic walk, which the
prefill tests pin to the per-token GEMV."""
import numpy as np
import pytest

from llamatov_amd import _lib, q8
from llamatov_amd import engine as dr
from llamatov_amd._lib import call

DYN, SLOT2, SLOT4, LS = range(4)
# N, K, T and the kernel of a device of 256 CUs
RULE = [
    # one block per leaf: always leaf-split
    (97, 32, 128, LS), (1000, 1024, 513, LS), (9728, 896, 129, LS), (9728, 896, 2048, LS),
    # two, in groups of two slots: 6.5 tiles per CU and round
    (11008, 2048, 128, LS), (11008, 2048, 192, SLOT2), (11008, 2048, 256, SLOT2), (11008, 2048, 257, LS),
    (11008, 2048, 300, SLOT2), (4096, 2048, 384, LS), (4096, 2048, 385, SLOT2),
    # two, not in groups: 10
    (2049, 1056, 129, LS), (1536, 1536, 1600, LS), (1536, 1536, 1729, DYN), (8960, 1536, 768, LS),
    (8960, 1536, 1024, DYN),
    # three to five: 128 tokens; 7 tiles (four slots), 8 (two slots, or five blocks), 9 (dynamic) per CU and round
    (896, 2080, 128, LS), (28672, 4096, 128, LS), (28672, 4096, 129, LS), (28672, 4096, 193, SLOT2),
    (4096, 4096, 416, LS), (4096, 4096, 417, SLOT4), (4096, 4096, 512, SLOT4), (4096, 4096, 513, SLOT2),
    (6144, 4096, 320, LS), (6144, 4096, 321, SLOT2), (6144, 4096, 512, SLOT2), (896, 4864, 2016, LS),
    (896, 4864, 2017, DYN), (896, 4864, 509, LS), (3584, 3584, 640, LS), (3584, 3584, 672, DYN),
    (8192, 5120, 224, LS), (8192, 5120, 256, DYN),
    # more: 64 tokens; 7 or 8 tiles per CU; groups of two slots for six blocks on a full chip only
    (33, 5152, 300, LS), (16384, 8192, 64, LS), (28672, 6144, 64, LS), (28672, 6144, 65, DYN),
    (28672, 6144, 97, SLOT2), (4096, 14336, 480, LS), (4096, 14336, 481, DYN), (8192, 8192, 192, LS),
    (8192, 8192, 193, SLOT4), (4096, 6144, 512, DYN), (4096, 6144, 768, SLOT2),
]


@pytest.mark.parametrize("N,K,T,kernel", RULE)
def test_choice(N, K, T, kernel, monkeypatch):
    for name in ("LS", "GROUPED"):
        monkeypatch.delenv(f"LT_GEMM_{name}", raising=False)
    assert _lib.raw("lt_q8_gemm_t_kernel")(256, T, N, K) == kernel


def test_choice_arguments(monkeypatch):
    kernel = _lib.raw("lt_q8_gemm_t_kernel")
    assert [kernel(*a) for a in ((0, 1, 1, 32), (256, 0, 1, 32), (256, 1, 0, 32), (256, 1, 1, 33))] == [-1] * 4
    monkeypatch.setenv("LT_GEMM_LS", "0")
    for walk, got in (("0", DYN), ("1", SLOT2), ("2", SLOT4)):
        monkeypatch.setenv("LT_GEMM_GROUPED", walk)
        assert kernel(256, 64, 4096, 4096) == got
    assert kernel(256, 64, 4096, 2048) == DYN       # (no four slots there)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,T", [r[:3] for r in RULE])
def test_default_kernel_equals_dynamic_walk(gpu, N, K, T, monkeypatch):
    print(f"[gpu-case] gemm rule N={N} K={K} T={T}", flush=True)
    rng = np.random.default_rng(N + K + T)
    rows = q8.quantize_rows((0.02 * rng.standard_normal((min(N, 1031), K))).astype(np.float32))
    rows = np.asarray(rows).reshape(min(N, 1031), -1)
    W = dr.DevTensor.from_host(np.ascontiguousarray(rows[np.arange(N) % len(rows)]), gpu)
    Wt = dr.DevTensor.empty((int(_lib.raw("lt_q8_tiles_bytes")(N, K)),), np.uint8, gpu)
    call("lt_q8_tiles", gpu.handle, W.vp, Wt.vp, N, K)
    x = dr.DevTensor.from_host(rng.standard_normal((T, K)).astype(np.float32), gpu)
    xq, xd = dr.DevTensor.empty((T * K,), np.int8, gpu), dr.DevTensor.empty((T * K // 32,), np.uint16, gpu)
    call("lt_quant_q8_bm", gpu.handle, x.vp, xq.vp, xd.vp, T, K)
    resid = dr.DevTensor.from_host(rng.standard_normal((T, N), dtype=np.float32), gpu)
    y = dr.DevTensor.empty((T, N), np.float32, gpu)

    def run():
        call("lt_q8_gemm_t", gpu.handle, Wt.vp, xq.vp, xd.vp, None, resid.vp, y.vp, T, N, K)
        return y.to_host().view(np.uint32)
    got = run()
    monkeypatch.setenv("LT_GEMM_LS", "0")
    monkeypatch.setenv("LT_GEMM_GROUPED", "0")
    assert np.array_equal(got, run())
    for t in (W, Wt, x, xq, xd, resid, y):
        t.free()


@pytest.mark.gpu
@pytest.mark.parametrize("F,K,T", [(4864, 896, 129), (4864, 896, 509), (96, 1024, 512), (32, 32, 500)])
def test_silu_with_quant_at_prompt_lengths(gpu, F, K, T):
    """The fused SiLU quant a narrow prefill takes past the batch sizes of a decode step, against the
    two launches."""
    print(f"[gpu-case] silu quant F={F} K={K} T={T}", flush=True)
    rng = np.random.default_rng(F + K + T)
    W = dr.DevTensor.from_host(q8.quantize_rows((0.1 * rng.standard_normal((2 * F, K))).astype(np.float32)), gpu)
    Wt = dr.DevTensor.empty((int(_lib.raw("lt_q8_tiles_bytes")(2 * F, K)),), np.uint8, gpu)
    call("lt_q8_tiles", gpu.handle, W.vp, Wt.vp, 2 * F, K)
    x = dr.DevTensor.from_host(rng.standard_normal((T, K)).astype(np.float32), gpu)
    q = [dr.DevTensor.empty((T * n,), np.int8, gpu) for n in (K, F, F)]
    d = [dr.DevTensor.empty((T * n // 32,), np.uint16, gpu) for n in (K, F, F)]
    v = dr.DevTensor.empty((T, F), np.float32, gpu)
    call("lt_quant_q8_bm", gpu.handle, x.vp, q[0].vp, d[0].vp, T, K)
    call("lt_q8_gemm_silu_t", gpu.handle, Wt.vp, q[0].vp, d[0].vp, v.vp, T, F, K)
    call("lt_quant_q8_bm", gpu.handle, v.vp, q[1].vp, d[1].vp, T, F)
    call("lt_q8_gemm_silu_quant_t", gpu.handle, Wt.vp, q[0].vp, d[0].vp, q[2].vp, d[2].vp, T, F, K)
    assert np.array_equal(q[1].to_host(), q[2].to_host()) and np.array_equal(d[1].to_host(), d[2].to_host())
    for t in (W, Wt, x, v, *q, *d):
        t.free()
