"""arc_attention_decode picks its launch shape (waves per workgroup, chunks per
split) from the context length and the kv heads: the contexts on both sides of
each line, few and many kv heads, against fp64 (per element 1e-3, the bar of the kernel) and
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


# (kv heads, query heads per kv head, T) and the shape the rule gives: both sides
# of each of its lines (2048, 3072, 4096 positions; 4, 24 and 32 kv heads; 96 and
# 256 workgroups of 8 waves)
LINES = [
    (4, 7, 2048, (4, 1)), (4, 7, 2049, (8, 1)), (24, 1, 2049, (8, 1)), (25, 1, 3072, (4, 1)), (25, 1, 3073, (8, 1)),
    (33, 1, 3073, (4, 1)), (3, 8, 3072, (4, 1)), (3, 8, 3073, (8, 1)), (8, 8, 4096, (8, 1)), (2, 7, 4097, (4, 1)),
    (4, 7, 4097, (4, 1)), (4, 7, 5888, (4, 1)), (4, 7, 5889, (8, 2)), (6, 8, 4097, (8, 2)), (8, 4, 8192, (8, 2)),
    (8, 4, 8193, (4, 1)), (12, 2, 5376, (8, 2)), (12, 2, 5377, (4, 1)), (7, 8, 9216, (8, 2)), (7, 8, 9217, (4, 1)),
    (4, 2, 32768, (8, 2)), (5, 2, 32768, (4, 1)),
]


@pytest.mark.parametrize("kv_heads,hpk,T,shape", LINES, ids=["%dx%d-%d" % c[:3] for c in LINES])
def test_rule(kv_heads, hpk, T, shape):
    """The automatic call gives the bits of the shape that the rule names (another
    shape adds in another order and differs in some), and is right."""
    n = kv_heads * hpk * 128
    kc = arc.synth_normal(SEED, 11, T * kv_heads * 128).astype(np.float16)
    vc = arc.synth_normal(SEED, 12, T * kv_heads * 128).astype(np.float16)
    q = arc.synth_normal(SEED, 13 + T, n) * np.float32(2.0)
    dk, dv, dq = dev(kc), dev(vc), dev(q)
    ws = arc.DeviceBuffer(arc.attention_workspace_bytes(kv_heads, hpk))
    got = {}
    for tune in ((0, 0), (4, 1), (8, 2 if T > 4096 else 1)):
        out = arc.DeviceBuffer(n * 4)
        arc.tune_attention(*tune)
        try:
            arc.attention_decode(dq, dk, dv, kv_heads, hpk, T, T, out, ws)
        finally:
            arc.tune_attention()
        got[tune] = out.download(np.uint32)
    for tune in list(got)[1:]:
        assert np.array_equal(got[0, 0], got[tune]) == (tune == shape), tune
    ref = orc.attention_decode_f64(q, kc, vc, T, kv_heads * hpk, kv_heads)
    assert orc.rel_err(got[0, 0].view(np.float32), ref) <= 1e-3


# the full grid of 64 splits and the plan's, on both sides of 4 kv heads and of 768 workgroups
@pytest.mark.parametrize("kv_heads,hpk,T", [(4, 1, 1), (5, 1, 1), (4, 7, 300), (5, 7, 300), (32, 2, 1536), (32, 2, 1537)])
def test_grid(kv_heads, hpk, T):
    n = kv_heads * hpk * 128
    kc = arc.synth_normal(SEED, 21, T * kv_heads * 128).astype(np.float16)
    vc = arc.synth_normal(SEED, 22, T * kv_heads * 128).astype(np.float16)
    q = arc.synth_normal(SEED, 23, n) * np.float32(2.0)
    out, ws = arc.DeviceBuffer(n * 4), arc.DeviceBuffer(arc.attention_workspace_bytes(kv_heads, hpk))
    got = []
    for _ in range(3):  # the workspace keeps what the call before left
        arc.attention_decode(dev(q), dev(kc), dev(vc), kv_heads, hpk, T, T, out, ws)
        got.append(out.download(np.float32))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    assert orc.rel_err(got[0], orc.attention_decode_f64(q, kc, vc, T, kv_heads * hpk, kv_heads)) <= 1e-3
