"""The prompt pass's tiled GEMM over several super-blocks: the hand-over from one
super-block to the next (codes and X in flight, counted waits) at every tile
height and format, with a last split that is shorter; and the rounding of the
decoded weights, bit for bit.

Bounds: per element 1e-3 with the floor 1e-3 * max|ref| against the fp16-operand
oracle, as for the other prompt-pass products."""
import numpy as np
import pytest

import arcllm_amd as arc
import oracle_lib as orc

pytestmark = pytest.mark.gpu

SEED = 0x57EAD
TOL = 1e-3
dev = arc.DeviceBuffer.from_array
HEIGHTS = [20, 64, 80, 96, 100, 128, 150, 192, 200, 256]  # inside and at the top of each tile


def packed(qtype, rows, K, stream):
    w = arc.synth_packed(arc.Q6_K if qtype == arc.Q6_K_PADDED else qtype, SEED, stream, rows, K)
    if qtype != arc.Q6_K_PADDED:
        return w, dev(w), qtype
    p = arc.DeviceBuffer(rows * (K // 256) * 212)
    arc.q6_pad(dev(w), rows, K, p)
    return w, p, arc.Q6_K


def x16(M, K, stream, scale=1.0):
    return (arc.synth_normal(SEED, stream, M * K) * np.float32(scale)).astype(np.float16).reshape(M, K)


def plan(N, K):
    """(splits, super-blocks per split) of the N x K product, from the size of its
    workspace: 256 fp16 rows of X and 256 fp32 rows of N per split."""
    sp = (arc.prefill_gemm_workspace_bytes(N, K) - 512 * K) // (1024 * N)
    return sp, -(-(K // 256) // sp)


def steady(N, K):
    sp, bps = plan(N, K)
    return sp >= 2 and bps >= 3 and 0 < K // 256 - (sp - 1) * bps < bps


def some(M):
    return sorted({0, M // 3, M // 2 + 1, M - 1})


@pytest.fixture(scope="module")
def weights():
    cache = {}

    def get(*key):
        if key not in cache:
            cache[key] = packed(*key)
        return cache[key]

    return get


@pytest.mark.parametrize("M", HEIGHTS)
@pytest.mark.parametrize("qtype", [arc.Q4_K, arc.Q6_K_PADDED])
def test_gemm(weights, qtype, M):
    N, K = 2432, 11008
    assert steady(N, K)
    w, dw, oq = weights(qtype, N, K, 1)
    x = x16(M, K, 2 + M)
    y, ws = arc.DeviceBuffer(M * N * 4), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gemm(qtype, dw, N, K, dev(x.view(np.uint16)), M, y, ws)
    got = y.download(np.float32).reshape(M, N)
    for m in some(M):
        assert orc.rel_err(got[m], orc.gemv_r64_f16(oq, w, N, K, x[m].astype(np.float64))) <= TOL, m


@pytest.mark.parametrize("M", HEIGHTS)
@pytest.mark.parametrize("v", [arc.Q4_K, arc.Q6_K_PADDED])
def test_qkv(weights, v, M):
    H, kvd, K = 1792, 256, 11008
    N = H + 2 * kvd
    assert steady(N, K)
    parts = [(0, weights(arc.Q4_K, H, K, 3), H), (H, weights(arc.Q4_K, kvd, K, 4), kvd), (H + kvd, weights(v, kvd, K, 5), kvd)]
    x = x16(M, K, 300 + M)
    y, ws = arc.DeviceBuffer(M * N * 4), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_qkv(parts[0][1][1], parts[1][1][1], parts[2][1][1], v, H, kvd, K, dev(x.view(np.uint16)), M, y, ws)
    got = y.download(np.float32).reshape(M, N)
    for m in some(M):
        for lo, (w, _, oq), rows in parts:
            ref = orc.gemv_r64_f16(oq, w, rows, K, x[m].astype(np.float64))
            assert orc.rel_err(got[m, lo:lo + rows], ref) <= TOL, (m, lo)


@pytest.mark.parametrize("M", HEIGHTS)
def test_gateup(weights, M):
    N, K = 200, 1280
    wg, dg, _ = weights(arc.Q4_K, N, K, 6)
    wu, du, _ = weights(arc.Q4_K, N, K, 7)
    x = x16(M, K, 600 + M, 0.05)
    s, ws = arc.DeviceBuffer(M * N * 2), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gateup(dg, du, N, K, dev(x.view(np.uint16)), M, s, ws)
    got = s.download(np.uint16).view(np.float16).reshape(M, N).astype(np.float64)
    for m in range(M):
        xm = x[m].astype(np.float64)
        ref = orc.swiglu_f64(orc.gemv_r64_f16(arc.Q4_K, wg, N, K, xm), orc.gemv_r64_f16(arc.Q4_K, wu, N, K, xm))
        assert orc.rel_err(got[m], ref) <= TOL, m


@pytest.mark.parametrize("N", [16384, 16385, 16500])  # past 16384 columns and 64 rows: 8 waves
@pytest.mark.parametrize("M", [64, 65, 96, 100, 150, 200, 256])
def test_gateup_wide(weights, N, M):
    K = 768
    wg, dg, _ = weights(arc.Q4_K, N, K, 11)
    wu, du, _ = weights(arc.Q4_K, N, K, 12)
    x = x16(M, K, 900 + M, 0.05)
    s, ws = arc.DeviceBuffer((M * N + 64) * 2), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    s.zero()
    arc.prefill_gateup(dg, du, N, K, dev(x.view(np.uint16)), M, s, ws)
    out = s.download(np.uint16)
    got = out[:M * N].view(np.float16).reshape(M, N).astype(np.float64)
    for m in some(M):
        xm = x[m].astype(np.float64)
        ref = orc.swiglu_f64(orc.gemv_r64_f16(arc.Q4_K, wg, N, K, xm), orc.gemv_r64_f16(arc.Q4_K, wu, N, K, xm))
        assert orc.rel_err(got[m], ref) <= TOL, m
    assert not out[M * N:].any(), "wrote past the result"


def q4_f64(w):
    """The exact weights of Q4_K blocks, [blocks, 256] in float64."""
    b = w.reshape(-1, 144)
    h = lambda a: b[:, a:a + 2].copy().view(np.float16).astype(np.float64)  # noqa: E731
    s = b[:, 4:16].astype(np.int64)
    sc = np.concatenate([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = np.concatenate([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    q = b[:, 16:].reshape(-1, 4, 1, 32).astype(np.int64)
    q = np.concatenate([q & 15, q >> 4], 2).reshape(-1, 8, 32)
    return ((h(0) * sc)[:, :, None] * q - (h(2) * mn)[:, :, None]).reshape(-1, 256)


@pytest.mark.parametrize("qtype", [arc.Q4_K, arc.Q6_K_PADDED])
def test_weights_round_to_fp32_then_fp16(qtype):
    """Rows of the identity as X give the decoded weights themselves: the element
    decode's fp32 value rounded to fp16, and not the exact value rounded once
    (which differs where the fp32 value is an fp16 tie; some of these are)."""
    N, K, M = 4096, 256, 256
    w, dw, oq = packed(qtype, N, K, 9)
    if qtype == arc.Q4_K:
        # in half of the blocks d * sc * q has up to 21 bits and dmin * mn lies below fp32's last
        b = w.reshape(-1, 144)
        d = (1 + np.arange(1, N, 2) % 1024 / 1024).astype(np.float16)
        b[::2, 0:2] = d.view(np.uint8).reshape(-1, 2)
        b[::2, 2:4] = [1, 0]  # 2^-24
        dw = dev(w)
    y, ws = arc.DeviceBuffer(M * N * 4), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gemm(qtype, dw, N, K, dev(np.eye(K, dtype=np.float16).view(np.uint16)), M, y, ws)
    got = y.download(np.float32).reshape(M, N).T
    want = orc.dequant(oq, w, N, K).reshape(N, K).astype(np.float16)
    assert np.array_equal(got, want.astype(np.float32))
    if qtype == arc.Q4_K:
        assert np.count_nonzero(q4_f64(w).astype(np.float16) != want) > 100
