"""arc_attention_decode picks its launch shape (waves per workgroup, chunks per
split) from the context length: the contexts on both sides of each line, few
and many kv heads, against fp64 (per element 1e-3, the bar of the kernel) and
against the shape of short contexts.  Two shapes differ only in the order of
fp32 sums of at most 6001 terms with weights that sum to 1: relative to the
largest output below 6001 * 2^-24 = 3.6e-4 at worst, some 1e-6 measured."""
import numpy as np
import pytest

import arcllm_amd as arc
import oracle_lib as orc

pytestmark = pytest.mark.gpu

SEED = 0xA77E5
dev = arc.DeviceBuffer.from_array


@pytest.mark.parametrize("T", [2047, 2048, 2049, 4096, 4097, 6001])
@pytest.mark.parametrize("kv_heads,hpk", [(1, 3), (3, 1), (4, 2)])
def test_shape_by_context(kv_heads, hpk, T):
    n = kv_heads * hpk * 128
    kc = arc.synth_normal(SEED, 1, T * kv_heads * 128).astype(np.float16)
    vc = arc.synth_normal(SEED, 2, T * kv_heads * 128).astype(np.float16)
    q = arc.synth_normal(SEED, 3 + T, n) * np.float32(2.0)
    dk, dv, dq = dev(kc), dev(vc), dev(q)
    ws = arc.DeviceBuffer(arc.attention_workspace_bytes(kv_heads, hpk))
    got = []
    for shape in ((0, 0), (4, 1)):
        out = arc.DeviceBuffer(n * 4)
        arc.tune_attention(*shape)
        try:
            for _ in range(2):  # the second call finds the counters of the first
                arc.attention_decode(dq, dk, dv, kv_heads, hpk, T, T, out, ws)
        finally:
            arc.tune_attention()
        got.append(out.download(np.float32))
    ref = orc.attention_decode_f64(q, kc, vc, T, kv_heads * hpk, kv_heads)
    assert orc.rel_err(got[0], ref) <= 1e-3
    assert np.max(np.abs(got[0] - got[1])) <= 3.6e-4 * np.max(np.abs(ref))
