"""The prompt pass's tiled GEMM at the edges of its tiles: row counts around
the 32 / 64 / 96 / 128 / 192 / 256-row tiles, column counts that are no multiple of a
tile, a vector store or 8, and one and several splits of K; every row and
column against the fp16-operand oracle.

Bound: per element 1e-3 with the floor 1e-3 * max|ref| (the bar of the other
prompt-pass products: operands are equal bit for bit, sums of K <= 2560
products in fp32 against fp64 leave < 1e-6 of max|ref|).  The fp16 SwiGLU
output adds its rounding (2^-11 relative)."""
import numpy as np
import pytest

import arcllm_amd as arc
import oracle_lib as orc

pytestmark = pytest.mark.gpu

SEED = 0x711E5
TOL = 1e-3
dev = arc.DeviceBuffer.from_array


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    assert arc.device_count() >= 1, "no HIP device visible"


def packed(qtype, rows, K, stream):
    w = arc.synth_packed(arc.Q6_K if qtype == arc.Q6_K_PADDED else qtype, SEED, stream, rows, K)
    if qtype != arc.Q6_K_PADDED:
        return w, dev(w), qtype
    p = arc.DeviceBuffer(rows * (K // 256) * 212)
    arc.q6_pad(dev(w), rows, K, p)
    return w, p, arc.Q6_K


def x16(M, K, stream, scale=1.0):
    return (arc.synth_normal(SEED, stream, M * K) * scale).astype(np.float16).reshape(M, K)


@pytest.mark.parametrize("M", [1, 31, 32, 33, 64, 65, 96, 97, 127, 128, 129, 192, 193, 255, 256])
@pytest.mark.parametrize("qtype,N,K", [(arc.Q4_K, 131, 2560), (arc.Q6_K_PADDED, 126, 256), (arc.Q6_K_PADDED, 257, 768)])
def test_gemm_tile_edges(qtype, N, K, M):
    w, dw, oq = packed(qtype, N, K, 1 + N)
    x = x16(M, K, 100 + M)
    y = arc.DeviceBuffer((M * N + 64) * 4)
    y.zero()
    ws = arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gemm(qtype, dw, N, K, dev(x.view(np.uint16)), M, y, ws)
    out = y.download(np.float32)
    got = out[:M * N].reshape(M, N)
    for m in range(M):
        ref = orc.gemv_r64_f16(oq, w, N, K, x[m].astype(np.float64))
        assert orc.rel_err(got[m], ref) <= TOL, m
    assert not out[M * N:].any(), "wrote past the result"


@pytest.mark.parametrize("M", [1, 32, 33, 65, 96, 97, 129, 192, 193, 256])
@pytest.mark.parametrize("N", [128, 200, 131])
def test_gateup_tile_edges(N, M):
    K = 512
    wg, dg, _ = packed(arc.Q4_K, N, K, 501)
    wu, du, _ = packed(arc.Q4_K, N, K, 502)
    x = x16(M, K, 600 + M, 0.05)
    s = arc.DeviceBuffer((M * N + 64) * 2)
    s.zero()
    ws = arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gateup(dg, du, N, K, dev(x.view(np.uint16)), M, s, ws)
    out = s.download(np.uint16)
    got = out[:M * N].view(np.float16).reshape(M, N).astype(np.float64)
    for m in range(M):
        xm = x[m].astype(np.float64)
        ref = orc.swiglu_f64(orc.gemv_r64_f16(arc.Q4_K, wg, N, K, xm), orc.gemv_r64_f16(arc.Q4_K, wu, N, K, xm))
        assert orc.rel_err(got[m], ref) <= TOL, m
    assert not out[M * N:].any(), "wrote past the result"


def test_gemm_takes_any_x_alignment():
    """X starting 2 bytes past a 16-byte boundary gives the same bits."""
    N, K, M = 256, 512, 40
    _, dw, _ = packed(arc.Q4_K, N, K, 7)
    x = x16(M, K, 8)
    ws = arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    got = []
    for off in (0, 1):
        buf = dev(np.concatenate([np.zeros(off, np.uint16), x.view(np.uint16).ravel(), np.zeros(8, np.uint16)]))
        y = arc.DeviceBuffer(M * N * 4)
        arc.prefill_gemm(arc.Q4_K, dw, N, K, buf.ptr + 2 * off, M, y, ws)
        got.append(y.download(np.uint32))
    assert np.array_equal(got[0], got[1])
