"""The tiled GEMM's choice of kernel (take_ls and the grouped walks in lt_prefill.hip): at both
sides of each line of the rule the default launch gives the bits of k_q8_gemm's dynamic walk, which
the prefill tests pin to the per-token GEMV."""
import numpy as np
import pytest

from llamatov_amd import _lib, q8
from llamatov_amd import engine as dr
from llamatov_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(97, 32), (9728, 896), (1000, 1024), (2049, 1056), (11008, 2048), (896, 2080),
                                 (896, 4864), (6144, 4096), (33, 5120), (33, 5152), (4096, 14336)])
@pytest.mark.parametrize("T", [128, 129, 300, 513])
def test_default_kernel_equals_dynamic_walk(gpu, N, K, T, monkeypatch):
    if N * K * T > 4 << 30:
        T = max(129, (4 << 30) // (N * K))
    print(f"[gpu-case] gemm rule N={N} K={K} T={T}", flush=True)
    rng = np.random.default_rng(N + K + T)
    W = dr.DevTensor.from_host(q8.quantize_rows((0.02 * rng.standard_normal((N, K))).astype(np.float32)), gpu)
    Wt = dr.DevTensor.empty((int(_lib.raw("lt_q8_tiles_bytes")(N, K)),), np.uint8, gpu)
    call("lt_q8_tiles", gpu.handle, W.vp, Wt.vp, N, K)
    x = dr.DevTensor.from_host(rng.standard_normal((T, K)).astype(np.float32), gpu)
    xq, xd = dr.DevTensor.empty((T * K,), np.int8, gpu), dr.DevTensor.empty((T * K // 32,), np.uint16, gpu)
    call("lt_quant_q8_bm", gpu.handle, x.vp, xq.vp, xd.vp, T, K)
    resid = dr.DevTensor.from_host(rng.standard_normal((T, N)).astype(np.float32), gpu)
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
