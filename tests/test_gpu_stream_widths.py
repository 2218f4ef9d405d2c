"""Decode batches of a few tokens: the stream kernels take their item width from
the row tiles there are (stream.hip, st_width).  Each case against the CPU
oracle, whose sums are binary64.

Tolerance: the products' error is that of the fp16 pair split (2^-22 a value)
and of fp32 sums of at most 64 blocks a wave and 4 waves; 3.4e-7 is seen at
H 2048, and 64 roundings of 2^-24 in a row are 4e-6.
"""
import numpy as np
import pytest

import oracle
import synth
from _util import gpu_context, moe_delta, rel_l2, upload_layer

pytestmark = pytest.mark.gpu

TOL = 4e-6


@pytest.mark.parametrize("T", [2, 3, 4, 5, 6, 8, 9, 11, 12, 16])
@pytest.mark.parametrize("shape", [
    dict(H=512, F=1792, E=32, K=4),     # 112 feature fragments: widths 2 .. 7 as T grows
    dict(H=2016, F=224, E=16, K=2),     # H not a multiple of any item width
    dict(H=1024, F=352, E=128, K=8),    # F not a multiple of any item width, many experts
], ids=lambda s: "H%(H)d_F%(F)d_E%(E)d" % s)
def test_stream_widths(shape, T):
    print("widths", shape, T, flush=True)
    L = synth.moe_layer(21 + T, **shape)
    x, hid = synth.activations(22, T, shape["H"])
    ctx = gpu_context()
    m = upload_layer(ctx, L)
    try:
        runs = [m.forward(x, hid) for _ in range(2)]
    finally:
        for t in m._keep:
            t.release()
        m.release()
    out, idx, w, probs = runs[0]
    np.testing.assert_array_equal(out, runs[1][0])   # the same bits from call to call
    r_out, r_idx, r_w, r_probs = oracle.moe_ffn(L, x, hid)
    np.testing.assert_array_equal(idx, r_idx)
    np.testing.assert_array_equal(w, r_w)
    err = rel_l2(moe_delta(out, hid), moe_delta(r_out, hid))
    print("rel_l2", err, flush=True)
    assert err < TOL, err


def test_stream_all_masked():
    """No row tiles at all: hidden stays as it is."""
    L = synth.moe_layer(5, H=512, F=224, E=8, K=2)
    x, hid = synth.activations(6, 3, 512)
    m = upload_layer(gpu_context(), L)
    try:
        out = m.forward(x, hid, mask=list(range(8)))[0]
    finally:
        for t in m._keep:
            t.release()
        m.release()
    np.testing.assert_array_equal(out, hid)
