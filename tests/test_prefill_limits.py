"""Largest K of the prompt-pass products.  Their tiles address X and 32 weight rows
with 32 bits: what lies past that is refused, and what lies below is right, also
where 128 weight rows (a workgroup's) take more than 4 GiB."""
import numpy as np
import pytest

import arcllm_amd as arc
import oracle_lib as orc

SEED = 0x1A26E


@pytest.mark.parametrize("M,K", [(1, (1 << 27) + 256), (32, 1 << 26), (33, 1 << 26), (256, 1 << 23), (256, 3 << 30)])
def test_too_large_is_refused(M, K):
    L, p = arc.lib(), 4096  # refused before any of the pointers is used
    for rc in (L.arc_prefill_gemm(arc.Q4_K, p, 128, K, p, M, p, p, None),
               L.arc_prefill_gateup(p, p, 128, K, p, M, p, p, None),
               L.arc_prefill_qkv(p, p, p, arc.Q4_K, 128, 128, K, p, M, p, p, None)):
        assert rc == 2 and b"2^31" in L.arc_last_error()


@pytest.mark.gpu
def test_weights_past_4_gib():
    nb, N = 160200, 128
    K, row = nb * 256, nb * 212
    assert N * row > 1 << 32
    rows, blocks = [0, 31, 32, 95, 127], [0, 77777, nb - 1]
    packed = arc.synth_packed(arc.Q6_K, SEED, 1, len(rows), 256 * len(blocks))
    x = (arc.synth_normal(SEED, 2, 256 * len(blocks))).astype(np.float16)
    w, xd = arc.DeviceBuffer(N * row), arc.DeviceBuffer(K * 2)
    w.zero()
    xd.zero()
    arc.synchronize()

    def put(at, a):
        a = np.ascontiguousarray(a)
        arc.check(arc.lib().arc_memcpy_htod(at, a.ctypes.data, a.nbytes, None))

    for i, r in enumerate(rows):
        for j, b in enumerate(blocks):
            put(w.ptr + r * row + b * 212, packed.reshape(len(rows), len(blocks), 210)[i, j])
    for j, b in enumerate(blocks):
        put(xd.ptr + b * 512, x[256 * j:256 * (j + 1)])
    y, ws = arc.DeviceBuffer(N * 4), arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    arc.prefill_gemm(arc.Q6_K_PADDED, w, N, K, xd, 1, y, ws)
    got = y.download(np.float32)
    want = np.zeros(N)
    want[rows] = orc.gemv_r64_f16(arc.Q6_K, packed, len(rows), 256 * len(blocks), x.astype(np.float64))
    # sums of 768 products that are not zero, in fp32
    assert np.max(np.abs(got - want)) <= 768 * 2.0 ** -24 * np.max(np.abs(want))
