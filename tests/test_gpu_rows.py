"""Q8_0 matrix times several rows (rows.hip) against binary64 sums.

Tolerance: activations enter exactly (three bf16 planes), so the error is that
of fp32 sums: at most ~60 roundings of 2^-24 in a row (16 blocks a level, the
levels, waves and segments), 3.6e-6 at worst and ~1e-7 as the roundings fall.
"""
import numpy as np
import pytest

import synth
from _util import gpu_context, rel_l2

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _dense(w, in_dim, out_dim):
    b = np.asarray(w).view(synth.Q8_DTYPE).reshape(out_dim, -1)
    m = b["qs"].astype(np.float64) * b["d"].astype(np.float64)[..., None]
    return m.reshape(out_dim, -1)[:, :in_dim]


def _case(in_dim, out_dim, rows, seed=0):
    rng = np.random.default_rng([in_dim, out_dim, rows, seed])
    w = synth.q8_0_tensor(rng, in_dim, out_dim)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    return w, x, x.astype(np.float64) @ _dense(w, in_dim, out_dim).T


@pytest.mark.parametrize("in_dim,out_dim,rows", [
    (2048, 200, 2), (2048, 200, 16),        # one 16-row tile, one column fragment
    (2048, 4100, 5),                        # two column fragments, partial last group
    (64, 32768, 3),                         # four column fragments
    (2048, 200, 17), (2048, 200, 32),       # two row fragments, last row of the row kernel
    (2048, 2100, 31),                       # two row x two column fragments
    (64, 8200, 32),                         # two row x four column fragments
    (1024, 70, 64),                         # rows x blocks at the GEMM's threshold ...
    (1024, 70, 65),                         # ... and past it: partial second row tile
    (2048, 31, 33), (7168, 129, 40),        # partial column groups, steps split over workgroups
    (2048, 1, 200),                         # a single output
    (96, 300, 700),                         # 3 blocks: an odd count, one segment
    (2080, 777, 130),                       # 65 blocks, odd output count
    (32, 40, 2100),                         # one block
    (512, 16500, 200),                      # 256-output groups
    (1000, 1501, 4), (1000, 1501, 20), (1000, 1501, 150),   # in_dim % 32 != 0, rows 16-byte aligned
    (2048, 16383, 1), (2048, 16384, 1), (64, 40000, 1),     # one row: either side of the rule
    (1001, 77, 9), (1003, 77, 40), (33, 300, 300),          # rows at any 4-byte alignment
    # either side of one round of the row kernel's tiles on 256 CUs: 16 x 16 outputs ...
    (64, 2048, 32), (64, 2049, 32), (64, 4096, 32), (64, 4097, 32),
    (512, 8192, 32), (512, 8193, 32), (64, 16384, 32), (64, 16385, 32),     # ... to 32 x 64
    (64, 1024, 500), (64, 1024, 520),                       # many rows of few blocks, and past one round
    (512, 8200, 33), (480, 8200, 33),                       # 16 blocks or fewer in several rounds
    (2048, 512, 100), (2080, 512, 100),                     # 64 blocks and 65
    (2080, 300, 20), (2080, 2100, 20), (2080, 300, 31),     # two row fragments of one and two columns
    (96, 8300, 300), (32, 8300, 300),                       # GEMM of an odd count of blocks, of one
    (2080, 70, 65), (4096, 31, 33),                         # GEMM: partial row and column tiles, split steps
    (896, 16384, 1), (895, 16400, 1), (864, 16384, 1),      # one row: 28 blocks and 27,
    (128, 65536, 1), (128, 65535, 1), (129, 65536, 1),      # 4 blocks and 5
])
def test_rows(in_dim, out_dim, rows):
    print("rows", in_dim, out_dim, rows, flush=True)
    w, x, ref = _case(in_dim, out_dim, rows)
    t = gpu_context().upload_q8_0(w, in_dim, out_dim)
    try:
        y = t.matvec(x)
    finally:
        t.release()
    assert np.isfinite(y).all()
    for r in range(rows):
        assert rel_l2(y[r], ref[r]) < TOL or out_dim == 1, (r, rel_l2(y[r], ref[r]))
    assert rel_l2(y, ref) < TOL


# in_dim not a multiple of 32, or rows off alignment, through every row kernel and GEMM that 256 CUs
# select: rows shorter than a block, of one block and a part, of a steady loop
# and a part.  x starts 0 or 4 bytes past a 16-byte boundary, between NaN that
# no sum may see.
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("in_dim,out_dim,rows", [(i, o, r) for i in (20, 40, 1100, 1120) for o, r in (
    (300, 1), (16500, 1),                               # a single row, aligned or not
    (300, 5), (4100, 5), (33000, 3),                    # row kernel, 16 rows: 1, 2, 4 fragments
    (300, 20), (2100, 20), (4200, 20), (8200, 20),      # ... one round of tiles
    (300, 120), (16500, 200),                           # ... GEMM of 256-output groups
)] + [(2100, 300, 20), (2100, 2100, 20),                # 32 rows: 1 and 2 fragments
      (2100, 300, 120), (40, 4200, 120)])               # GEMM of 128-output groups
def test_rows_ragged(in_dim, out_dim, rows, off):
    import torch
    print("ragged", in_dim, out_dim, rows, off, flush=True)
    w, x, ref = _case(in_dim, out_dim, rows, 3)
    buf = torch.full((rows * in_dim + 8,), float("nan"), device="cuda")
    xd = buf[off:off + rows * in_dim]
    xd.copy_(torch.from_numpy(x).reshape(-1))
    y = torch.full((rows, out_dim), float("nan"), device="cuda")
    torch.cuda.synchronize()
    ctx = gpu_context()
    t = ctx.upload_q8_0(w, in_dim, out_dim)
    try:
        t.matvec_dev(xd.data_ptr(), y.data_ptr(), rows)
        ctx.synchronize()
    finally:
        t.release()
    y = y.cpu().numpy()
    assert np.isfinite(y).all()
    for r in range(rows):
        assert rel_l2(y[r], ref[r]) < TOL, (r, rel_l2(y[r], ref[r]))


@pytest.mark.parametrize("in_dim,out_dim,rows", [
    (512, 96, 8), (512, 96, 24), (2048, 96, 80), (1000, 96, 80),
    (4096, 96, 80), (2100, 96, 80), (512, 16500, 200),      # GEMM: split steps, ragged, 256-output groups
])
def test_rows_special_values(in_dim, out_dim, rows):
    """Infinities, NaN and large or small rows stay with their own row; a
    power of two on a row is a power of two on its result."""
    w, x, ref = _case(in_dim, out_dim, rows, 1)
    x[1] *= np.float32(2.0 ** 100)
    x[2] *= np.float32(2.0 ** -80)
    x[3, 7] = np.inf
    x[4, in_dim - 1] = -np.inf
    x[5, 40] = np.nan
    x[6, 3] = np.array([0x7f800001], np.uint32).view(np.float32)[0]   # a NaN with only a low payload bit
    t = gpu_context().upload_q8_0(w, in_dim, out_dim)
    try:
        y = t.matvec(x)
    finally:
        t.release()
    q = np.asarray(w).view(synth.Q8_DTYPE).reshape(out_dim, -1)["qs"].reshape(out_dim, -1)
    for r, k, s in ((3, 7, 1.0), (4, in_dim - 1, -1.0)):
        want = np.where(q[:, k] == 0, np.nan, np.where(q[:, k] > 0, s, -s) * np.inf)
        np.testing.assert_array_equal(y[r], want.astype(np.float32))
    assert np.isnan(y[5]).all() and np.isnan(y[6]).all()
    ref[1] *= 2.0 ** 100
    ref[2] *= 2.0 ** -80
    for r in [0, 1, 2] + list(range(7, rows)):
        assert rel_l2(y[r], ref[r]) < TOL, r


@pytest.mark.parametrize("in_dim,out_dim,rows", [
    (512, 96, 16), (2048, 300, 24),         # row kernel: one and two row fragments
    (2048, 4200, 12), (64, 33000, 12), (64, 8200, 24),      # ... two and four column fragments
    (2048, 96, 100), (2048, 8200, 24),      # ... one round of tiles
    (4096, 96, 100), (512, 16500, 200),     # GEMM: steps split over workgroups, 256-output groups
    (1000, 300, 24), (1000, 300, 120), (2100, 300, 120),    # in_dim % 32 != 0
])
def test_rows_range(in_dim, out_dim, rows):
    """Rows of every magnitude that fp32 holds, subnormals included, up to
    where 32 unscaled products would leave it; rows beside them keep the bits
    they have without them.  A result below 2^-126 is rounded at 2^-149 once per
    wave and segment: at most 16 such roundings."""
    rng = np.random.default_rng([in_dim, out_dim, rows, 9])
    w = synth.q8_0_tensor(rng, in_dim, out_dim)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    ctx = gpu_context()
    t = ctx.upload_q8_0(w, in_dim, out_dim)
    try:
        plain = t.matvec(x)
        exps = [-145, -135, -126, -120, -112, -100, -70, -62, 112, 116, 119]
        for r, e in enumerate(exps):
            x[r] = (x[r].astype(np.float64) * 2.0 ** e).astype(np.float32)
        y = t.matvec(x)
    finally:
        t.release()
    ref = x.astype(np.float64) @ _dense(w, in_dim, out_dim).T
    assert np.abs(ref).max() < 2.0 ** 127
    for r, e in enumerate(exps):
        err = np.linalg.norm(y[r].astype(np.float64) - ref[r])
        bound = TOL * np.linalg.norm(ref[r]) + 16 * 2.0 ** -149 * np.sqrt(out_dim)
        assert err < bound, (e, err / np.linalg.norm(ref[r]))
    np.testing.assert_array_equal(y[len(exps):], plain[len(exps):])


@pytest.mark.parametrize("in_dim", [2048, 4096])   # row kernel; GEMM, its steps split over workgroups
def test_rows_captured(in_dim):
    """A recorded call needs nothing the context did not already hold, and
    replays to the eager result."""
    import torch
    ctx = gpu_context()
    out_dim, rows = 512, 100
    w, x, _ = _case(in_dim, out_dim, rows, 2)
    t = ctx.upload_q8_0(w, in_dim, out_dim)
    xd = torch.from_numpy(x).cuda()
    y0, y1 = (torch.zeros((rows, out_dim), device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    ctx.capture_begin()
    t.matvec_dev(xd.data_ptr(), y1.data_ptr(), rows)
    g = ctx.capture_end()
    try:
        t.matvec_dev(xd.data_ptr(), y0.data_ptr(), rows)
        ctx.synchronize()
        for _ in range(3):
            y1.zero_()
            torch.cuda.synchronize()
            g.launch()
            ctx.synchronize()
            assert torch.equal(y0, y1)
    finally:
        g.release()
        t.release()
