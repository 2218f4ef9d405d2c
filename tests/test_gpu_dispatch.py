"""The dispatch of many pairs over several workgroups (grouped.hip): pair counts
at the edges of a share, of the workgroup limit and of a pass of loads, with and
without masked experts, against the CPU oracle.

Tolerance: the fp32 path's (pair-split products, fp32 sums; 3.4e-7 is seen at
H 2048): 64 roundings of 2^-24 are 4e-6.
"""
import numpy as np
import pytest

import oracle
import synth
from _util import gpu_context, moe_delta, rel_l2, upload_layer

pytestmark = pytest.mark.gpu

TOL = 4e-6


def _check(L, T, mask, sel):
    x, hid = synth.activations(32, T, 64)
    ctx = gpu_context()
    m = upload_layer(ctx, L)
    ctx.set_mfma_min_tokens(0)
    try:
        out, idx, w, probs = m.forward(x, hid, mask=mask)
    finally:
        ctx.set_mfma_min_tokens(512)
        for t in m._keep:
            t.release()
        m.release()
    r_out, r_idx, r_w, _ = oracle.moe_ffn(L, x[sel], hid[sel], mask=mask)
    np.testing.assert_array_equal(idx[sel], r_idx)
    np.testing.assert_array_equal(w[sel], r_w)
    got, want = moe_delta(out, hid), moe_delta(r_out, hid[sel])
    assert np.isfinite(got).all()
    assert rel_l2(got[sel], want) < TOL
    # no row lost: a row of no contribution is one whose experts are all masked
    dead = ~np.any(got != 0, axis=1)
    none = np.isin(idx, mask).all(axis=1) if mask else np.zeros(T, bool)
    np.testing.assert_array_equal(dead, none)


@pytest.mark.parametrize("mask", [None, [0, 3]], ids=["all", "masked"])
@pytest.mark.parametrize("T", [170, 171, 341, 342, 1000, 2730, 2731, 4096, 4100])
def test_dispatch_shares(T, mask):
    print("dispatch", T, mask, flush=True)
    sel = np.unique(np.concatenate([np.arange(0, T, max(1, T // 97)), [T - 1, T // 2]]))
    _check(synth.moe_layer(31, H=64, F=64, E=8, K=3), T, mask, sel)


@pytest.mark.parametrize("mask", [None, [0, 3]], ids=["all", "masked"])
@pytest.mark.parametrize("T", [2048, 2049, 3000, 4096])
def test_dispatch_chunks(T, mask):
    """More pairs than one pass of loads holds (16384): exactly one, one and 8
    pairs, shares that straddle the edge, two whole ones.  Every row is compared,
    so that one slot lost or handed out twice shows (~5e-3 of the whole)."""
    print("dispatch chunks", T, mask, flush=True)
    _check(synth.moe_layer(33, H=64, F=64, E=16, K=8), T, mask, np.arange(T))
