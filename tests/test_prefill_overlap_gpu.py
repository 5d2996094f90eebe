"""The prompt-pass products read X where the caller has it.  Where X shares
memory with what the launch itself writes (arc_prefill_gateup's s, the split
partials in the workspace) they take a copy first: the same bits as with separate
buffers."""
import numpy as np
import pytest

import arcllm_amd as arc

pytestmark = pytest.mark.gpu

SEED = 0x0E41A
dev = arc.DeviceBuffer.from_array


def x16(M, K):
    return (arc.synth_normal(SEED, 1, M * K) * np.float32(0.05)).astype(np.float16).view(np.uint16)


def q4(N, K, stream):
    return dev(arc.synth_packed(arc.Q4_K, SEED, stream, N, K))


# where s starts in halves from x: on it, inside it, before it with an overlap of
# one half, and at an odd half
@pytest.mark.parametrize("at", [0, 512 * 7, 1 - 200 * 512, -333])
@pytest.mark.parametrize("M", [40, 200])
def test_gateup_over_its_input(M, at):
    N = K = 512  # s as large as x
    g, u, x = q4(N, K, 2), q4(N, K, 3), x16(M, K)
    at = max(at, 1 - M * K)
    ws = arc.DeviceBuffer(arc.prefill_gemm_workspace_bytes(N, K))
    s = arc.DeviceBuffer(M * N * 2)
    arc.prefill_gateup(g, u, N, K, dev(x), M, s, ws)
    want = s.download(np.uint16)
    first = max(0, -at)  # of x, in halves; x stays 16-byte aligned
    first = (first + 7) // 8 * 8
    both = dev(np.concatenate([np.zeros(first, np.uint16), x, np.zeros(M * N, np.uint16)]))
    arc.prefill_gateup(g, u, N, K, both.ptr + 2 * first, M, both.ptr + 2 * (first + at), ws)
    got = both.download(np.uint16)[first + at:first + at + M * N]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("qkv", [False, True])
def test_input_among_the_partials(qkv):
    M, K, N = 40, 512, 512
    x, w = x16(M, K), q4(N, K, 2)
    nbytes = arc.prefill_gemm_workspace_bytes(N, K)

    def run(xp, ws):
        y = arc.DeviceBuffer(M * N * 4)
        if qkv:
            arc.prefill_qkv(w, w.ptr + 256 * (K // 256) * 144, w.ptr + 384 * (K // 256) * 144, arc.Q4_K, 256, 128, K, xp, M, y,
                            ws)
        else:
            arc.prefill_gemm(arc.Q4_K, w, N, K, xp, M, y, ws)
        return y.download(np.uint32)

    ws = arc.DeviceBuffer(nbytes)
    want = run(dev(x), ws)
    host = np.zeros(nbytes // 2, np.uint16)
    host[256 * K:256 * K + M * K] = x  # the partials follow 256 rows of X
    inside = dev(host)
    assert np.array_equal(run(inside.ptr + 2 * 256 * K, inside), want)
