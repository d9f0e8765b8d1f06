"""The tile kernel of the projections (linear_tile.hip) at its edges: row and
column remainders of every tile shape, K tails, K split over workgroups, the
three weight types, infinities, and a first call under graph capture.

Bound per output, against float64: the sum's f32 rounding (K + 8 roundings of
at most 2^-24 of the sum of |x w|), plus, for bf16 weights with K % 32 == 0, what
two bf16 pieces leave of x (2^-17 of each product).
"""
import numpy as np
import pytest

import spissa_amd as sa
from spissa_amd.linear import DTYPE_BF16, DTYPE_F16, DTYPE_F32, StreamingLinearConfig
from spissa_amd.synth import normal_f32, seed_for
from tests.helpers import assert_bitwise

pytestmark = pytest.mark.gpu


def make(m, n, k, dtype, bias=True):
    w = normal_f32(seed_for(71, m, n, "q", k), n * k, 0.0, 0.05)
    x = normal_f32(seed_for(71, m, n, "k", k), m * k)
    b = normal_f32(seed_for(71, m, n, "v", k), n) if bias else None
    if dtype == DTYPE_F32:
        return w, w.astype(np.float64), x, b
    if dtype == DTYPE_F16:
        h = w.astype(np.float16)
        return h.view(np.uint16).copy(), h.astype(np.float64), x, b
    u = w.view(np.uint32)
    bits = ((u.astype(np.uint64) + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return bits, (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64), x, b


def check(got, w64, x, b, m, n, k, dtype):
    x64, w64 = x.reshape(m, k).astype(np.float64), w64.reshape(n, k)
    ref = x64 @ w64.T + (0 if b is None else b.astype(np.float64))
    mag = np.abs(x64) @ np.abs(w64).T + (0 if b is None else np.abs(b.astype(np.float64)))
    eps = (k + 8) * 2.0 ** -24 + (2.0 ** -17 if dtype == DTYPE_BF16 and k % 32 == 0 else 0.0)
    worst = float(np.max(np.abs(got.reshape(m, n) - ref) / (eps * mag)))
    print(f"[tile] {m} x {n} x {k} dtype {dtype}: {worst:.3f} of the bound", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("m,n,k", [
    (5, 4096, 64),      # two k tiles (bf16: the skinny kernel)
    (33, 130, 3072),    # one row and two columns past a tile, K split 16 ways
    (31, 127, 1000),    # K tail of 8, split 8 ways
    (65, 1153, 2048),   # split 6 or 8 ways
    (129, 2050, 1336),  # K tail of 24, split 3 ways
    (700, 2047, 96),    # 64-row tiles; three k tiles: no whole round of the ring
    (1030, 1500, 160),  # 64-row tiles, several per CU
])
def test_tile_edges(gpu, dtype, m, n, k):
    w, w64, x, b = make(m, n, k, dtype)
    got = sa.linear(sa.LinearWeight(w, dtype, n, k), x, b, StreamingLinearConfig(m, k, n))
    check(got, w64, x, b, m, n, k, dtype)


# (dtype, m, n, k, rows and columns of the tile, whether K is split): every tile
# shape of every form of the kernel, with and without the merge, ragged in both
# directions, the smallest sizes that take it
EVERY_TILE = [
    (DTYPE_BF16, 241, 34, 128, 32, 128, False),
    (DTYPE_BF16, 19, 75, 736, 32, 128, True),
    (DTYPE_BF16, 3501, 386, 32, 64, 128, False),
    (DTYPE_BF16, 851, 33, 2368, 64, 128, True),
    (DTYPE_BF16, 3604, 776, 96, 128, 128, False),
    (DTYPE_BF16, 3145, 32, 2272, 128, 128, True),
    (DTYPE_BF16, 769, 6469, 224, 128, 256, False),
    (DTYPE_BF16, 2724, 668, 2816, 128, 256, True),
    (DTYPE_BF16, 22, 662, 72, 32, 128, False),  # K % 32 != 0: three pieces of x
    (DTYPE_BF16, 19, 92, 600, 32, 128, True),
    (DTYPE_BF16, 581, 2722, 24, 64, 128, False),
    (DTYPE_BF16, 1014, 34, 1576, 64, 128, True),
    (DTYPE_BF16, 2884, 1036, 40, 128, 128, False),
    (DTYPE_BF16, 2525, 36, 2504, 128, 128, True),
    (DTYPE_BF16, 1292, 5027, 72, 128, 256, False),
    (DTYPE_BF16, 199, 5435, 3624, 128, 256, True),
    (DTYPE_F16, 22, 662, 72, 32, 128, False),
    (DTYPE_F16, 23, 100, 456, 32, 128, True),
    (DTYPE_F16, 2749, 258, 40, 64, 128, False),
    (DTYPE_F16, 2494, 33, 504, 64, 128, True),
    (DTYPE_F16, 3664, 525, 40, 128, 128, False),
    (DTYPE_F16, 2786, 33, 1128, 128, 128, True),
    (DTYPE_F32, 185, 109, 52, 32, 128, False),
    (DTYPE_F32, 22, 36, 1324, 32, 128, True),
    (DTYPE_F32, 2749, 258, 36, 64, 128, False),
    (DTYPE_F32, 2494, 33, 508, 64, 128, True),
    (DTYPE_F32, 3337, 642, 28, 128, 128, False),
    (DTYPE_F32, 1826, 33, 1572, 128, 128, True),
]


@pytest.mark.parametrize("dtype,m,n,k,rows,columns,split", EVERY_TILE)
def test_every_tile_shape(gpu, dtype, m, n, k, rows, columns, split):
    from spissa_amd import _ffi
    from spissa_amd.device import plan_linear

    p = plan_linear(dtype, m, n, k)
    assert (p["path"], p["tile_rows"], p["tile_columns"], p["splits"] > 1) == (_ffi.LINEAR_TILE, rows, columns, split)
    w, w64, x, b = make(m, n, k, dtype)
    for bias in (b, None):
        got = sa.linear(sa.LinearWeight(w, dtype, n, k), x, bias, StreamingLinearConfig(m, k, n))
        check(got, w64, x, bias, m, n, k, dtype)


@pytest.mark.parametrize("m,n,k,splits", [
    (40, 256, 256, 1),
    (33, 130, 3072, 16),  # formed again where the partial sums are merged
])
@pytest.mark.parametrize("dtype", [DTYPE_F16, DTYPE_F32])
def test_infinities_keep_the_reference_result(gpu, dtype, m, n, k, splits):
    """An infinite activation, or one that rounds up to infinity in bf16, splits
    into pieces of both signs; such outputs equal the in-order sum. Subnormal
    f16 weights are exact."""
    from spissa_amd.device import plan_linear

    assert plan_linear(dtype, m, n, k)["splits"] == splits
    w, w64, x, b = make(m, n, k, dtype)
    x = x.reshape(m, k).copy()
    x[3, 7] = np.inf
    x[5, 9] = -np.inf
    x[5, 200] = np.inf
    x[8, 1] = 3.4e38
    x[11, 0] = np.nan
    if dtype == DTYPE_F16:
        w = w.copy()
        w[:k] = 1  # row 0: the smallest subnormal
        w64 = w.view(np.float16).astype(np.float64)
    got = sa.linear(sa.LinearWeight(w, dtype, n, k), x.ravel(), b, StreamingLinearConfig(m, k, n)).reshape(m, n)
    with np.errstate(all="ignore"):
        w32 = w64.reshape(n, k).astype(np.float32)
        ref = np.broadcast_to(b, (m, n)).astype(np.float32).copy()
        for i in range(k):  # the reference's order, each product rounded
            ref = (ref + (x[:, i:i + 1] * w32[:, i]).astype(np.float32)).astype(np.float32)
    odd = ~np.isfinite(x).all(axis=1)
    assert np.array_equal(np.isnan(got[odd]), np.isnan(ref[odd]))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf]) and np.array_equal(np.isinf(got), inf)
    # the finite outputs of the finite rows, the one of the largest value included
    # (a row with an infinite output is compared above)
    fine = ~odd & ~inf.any(axis=1)
    check(got[fine], w64, x[fine].ravel(), b, int(fine.sum()), n, k, dtype)
    at = np.flatnonzero(np.isfinite(ref[8]))
    check(got[8, at], w64.reshape(n, k)[at], x[8], b[at], 1, at.size, k, dtype)


@pytest.mark.parametrize("dtype", [DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("m,n,k", [(40, 256, 2048), (333, 130, 1000), (6, 520, 4096)])
def test_rows_of_a_wide_range_keep_their_small_values(gpu, dtype, m, n, k):
    """Rows whose largest values meet weights of zero (pruned columns): the
    outputs are the small values' sums, at the bound of their own products."""
    w, _, x, b = make(m, n, k, dtype)
    w, x = w.reshape(n, k).copy(), x.reshape(m, k).copy()
    pruned = [3, k // 2, k - 1]
    w[:, pruned] = 0
    x[:, pruned] = 0.0
    for i, big in enumerate((1e5, 1e7, 1e8, -1e10, 2.0 ** 40, 1e20, -1e30)):
        if i < m:
            x[i::7, pruned[i % 3]] = big
    x[1::7] *= np.float32(1e-20)  # (1e-13 beside values of 1e-20)
    half = np.float32(2.0 ** -23)  # two levels: half the columns far below the other half, which this row of w ignores
    x[2::7, : k // 2] *= half
    w[n // 2, k // 2 :] = 0
    w64 = (w.view(np.float16) if dtype == DTYPE_F16 else w).astype(np.float64)
    got = sa.linear(sa.LinearWeight(w.ravel(), dtype, n, k), x.ravel(), b, StreamingLinearConfig(m, k, n))
    check(got, w64, x.ravel(), b, m, n, k, dtype)
    got = sa.linear(sa.LinearWeight(w.ravel(), dtype, n, k), x.ravel(), None, StreamingLinearConfig(m, k, n))
    check(got, w64, x.ravel(), None, m, n, k, dtype)


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("m,n,k", [
    (33, 1000, 40),      # K % 32 != 0 throughout
    (33, 130, 3080),
    (129, 2050, 1336),
    (700, 2047, 104),
    (1500, 5110, 72),
])
def test_no_bit_of_x_is_dropped(gpu, dtype, m, n, k):
    """Weight rows with a single 1: the outputs are the activations themselves,
    all 24 bits of them, where the sums are in whole f32 products (the pieces of
    one value add up in f32 without rounding, and zeros add nothing)."""
    x = normal_f32(seed_for(73, m, n, "k", k), m * k).reshape(m, k)
    x *= (2.0 ** np.linspace(-60, 60, m)).astype(np.float32)[:, None]
    col = np.random.RandomState(m + n).randint(0, k, n)
    w = np.zeros((n, k), np.float32)
    w[np.arange(n), col] = 1.0
    if dtype == DTYPE_F16:
        w = w.astype(np.float16).view(np.uint16)
    elif dtype == DTYPE_BF16:
        w = (w.view(np.uint32) >> 16).astype(np.uint16)
    got = sa.linear(sa.LinearWeight(np.ascontiguousarray(w).ravel(), dtype, n, k), x.ravel(), None,
                    StreamingLinearConfig(m, k, n))
    assert_bitwise(got.reshape(m, n), x[:, col], "selected activations")


def test_first_call_under_capture(gpu):
    """The plan is a matter of the sizes alone: a session's first call, captured,
    shares K over workgroups as an eager one does, and gives its bits."""
    import torch

    from spissa_amd.device import Session, plan_linear

    m, n, k = 24, 512, 2048
    assert plan_linear(DTYPE_BF16, m, n, k)["splits"] == 16
    w, w64, x, _ = make(m, n, k, DTYPE_BF16, bias=False)
    st = torch.cuda.Stream()
    s = Session(0, stream=st)
    lw = s.linear_weight(w, DTYPE_BF16, n, k)
    dx = torch.from_numpy(x).cuda()
    out = torch.zeros(m * n, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        s.linear(lw, dx, None, m, out)
    first = None
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        check(got, w64, x, None, m, n, k, DTYPE_BF16)
        if first is not None:
            assert_bitwise(got, first, "replay")
        first = got
    with torch.cuda.stream(st):
        s.linear(lw, dx, None, m, out)
    s.sync()
    assert_bitwise(out.cpu().numpy(), first, "eager after the replays")


@pytest.mark.parametrize("m,n,k", [
    (5, 1, 128),        # one row, one k step a wave
    (8, 511, 1280),     # ten steps: a round of eight and two more
    (16, 17, 512),      # one row past a block, the longest K at 16 tokens
    (17, 130, 1024),    # the second block's first token, whole rounds of eight steps
    (32, 8191, 384),    # three steps a wave
    (33, 4095, 640),    # five steps: a round of four and one more
    (64, 200, 512),
])
def test_short_k(gpu, m, n, k):
    from spissa_amd import _ffi
    from spissa_amd.device import plan_linear

    assert plan_linear(DTYPE_BF16, m, n, k)["path"] == _ffi.LINEAR_SHORT
    w, w64, x, b = make(m, n, k, DTYPE_BF16)
    got = sa.linear(sa.LinearWeight(w, DTYPE_BF16, n, k), x, b, StreamingLinearConfig(m, k, n))
    check(got, w64, x, b, m, n, k, DTYPE_BF16)


@pytest.mark.parametrize("m,n,k,rows,columns", [
    (4090, 5110, 1056, 256, 320),  # ragged both ways, an odd number of k tiles
    (4090, 5110, 1024, 256, 320),
    (4085, 8190, 96, 128, 256),    # odd
    (2050, 16300, 64, 128, 256),
    (4000, 8200, 32, 128, 256),    # one k tile
])
def test_prompt_tiles(gpu, m, n, k, rows, columns):
    from spissa_amd import _ffi
    from spissa_amd.device import plan_linear

    p = plan_linear(DTYPE_BF16, m, n, k)
    assert (p["path"], p["tile_rows"], p["tile_columns"]) == (_ffi.LINEAR_GEMM, rows, columns)
    w, w64, x, b = make(m, n, k, DTYPE_BF16)
    for bias in (b, None):
        got = sa.linear(sa.LinearWeight(w, DTYPE_BF16, n, k), x, bias, StreamingLinearConfig(m, k, n))
        check(got, w64, x, bias, m, n, k, DTYPE_BF16)


@pytest.mark.parametrize("m,n,k,path", [
    (5, (1 << 21) + 5, 32, "gemm"),
    (5, (1 << 21) + 5, 128, "short"),
    (5, (1 << 21) + 5, 544, "skinny"),
    (17, 1 << 21, 32, "tile"),            # the longest rows the tile kernel takes
    (259, (1 << 21) + 5, 32, "gemm"),     # stored with 64-bit addresses, ragged both ways
    (17, 40, 1 << 21, "tile"),
    (17, 40, (1 << 21) + 32, "gemm"),     # an odd number of k tiles
])
def test_rows_past_the_32_bit_offsets(gpu, m, n, k, path):
    from spissa_amd import _ffi
    from spissa_amd.device import plan_linear

    assert plan_linear(DTYPE_BF16, m, n, k)["path"] == getattr(_ffi, f"LINEAR_{path.upper()}")
    rng = np.random.default_rng(m + k)
    w = (rng.standard_normal(n * k, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    x, b = rng.standard_normal(m * k, np.float32), rng.standard_normal(n, np.float32)
    got = sa.linear(sa.LinearWeight(w, DTYPE_BF16, n, k), x, b, StreamingLinearConfig(m, k, n)).reshape(m, n)
    rows = sorted({0, 1, m // 2, m - 2, m - 1})
    cols = np.unique(np.r_[0:40, n // 2:n // 2 + 40, n - 340:n])
    cols = cols[(cols >= 0) & (cols < n)]
    w64 = (w.reshape(n, k)[cols].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    check(got[np.ix_(rows, cols)], w64, x.reshape(m, k)[rows], b[cols], len(rows), len(cols), k, DTYPE_BF16)
    # every other row and column, by its sums: the x (and bias) sums against the weights
    if k <= 128:
        w32 = (w.astype(np.uint32) << 16).view(np.float32).reshape(n, k)
        ref = w32 @ x.reshape(m, k).T.astype(np.float32) + b[:, None]
        assert np.max(np.abs(got.T - ref)) <= 1e-4 * np.max(np.abs(ref))


def test_threads_share_a_session(gpu):
    """Projections whose K is split, from several threads on one session: each
    call's partial sums are its own until its result is formed."""
    import threading

    import torch

    from spissa_amd.device import Session, plan_linear

    st = torch.cuda.Stream()
    s = Session(0, stream=st)
    jobs = []
    for dtype, m, n, k in [(DTYPE_BF16, 24, 512, 2048), (DTYPE_F16, 33, 130, 3072), (DTYPE_F32, 40, 256, 2048),
                           (DTYPE_BF16, 31, 520, 4000)]:
        assert plan_linear(dtype, m, n, k)["splits"] > 1
        w, w64, x, _ = make(m, n, k, dtype, bias=False)
        jobs.append((s.linear_weight(w, dtype, n, k), torch.from_numpy(x).cuda(),
                     [torch.empty(m * n, device="cuda") for _ in range(50)], (w64, x, None, m, n, k, dtype)))
    torch.cuda.synchronize()
    failed = []

    def work(lw, dx, outs, case):
        try:
            for out in outs:
                s.linear(lw, dx, None, case[3], out)
        except Exception as e:  # shown by the main thread
            failed.append(e)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    s.sync()
    assert not failed, failed
    for _, _, outs, (w64, x, b, m, n, k, dtype) in jobs:
        first = outs[0].cpu().numpy()
        check(first, w64, x, b, m, n, k, dtype)
        for out in outs[1:]:
            assert_bitwise(out.cpu().numpy(), first, "a repeated call")


@pytest.mark.parametrize("m,n,k", [
    (5, 1, 64),        # one row, one k tile for one wave
    (16, 17, 96),      # one row past a block, half a k tile
    (9, 4096, 544),    # the most rows of 16-row workgroups, ragged waves
    (16, 4097, 1152),  # 32-row workgroups, one row past a block
])
def test_up_to_16_tokens(gpu, m, n, k):
    w, w64, x, b = make(m, n, k, DTYPE_BF16)
    got = sa.linear(sa.LinearWeight(w, DTYPE_BF16, n, k), x, b, StreamingLinearConfig(m, k, n))
    check(got, w64, x, b, m, n, k, DTYPE_BF16)


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [
    (1, 8),         # one row, one piece
    (4096, 520),    # a lane past 64 pieces, the last size of one row per wave at 3 and 4 tokens
    (4097, 1544),   # one row past it, four pieces a lane, the last of them in one lane
    (130, 2560),
    (3075, 3072),
    (35, 3080),     # a seventh piece, in one lane
    (130, 4096),    # the longest row in one pass
    (35, 4104),     # and one piece more
    (2048, 512),    # the most rows of one piece a lane that are in flight whole
    (2049, 504),    # one row past them
    (16385, 256),   # where three and four tokens take two rows a wave
])
def test_few_token_rows(gpu, dtype, m, n, k):
    w, w64, x, b = make(m, n, k, dtype)
    got = sa.linear(sa.LinearWeight(w, dtype, n, k), x, b, StreamingLinearConfig(m, k, n))
    check(got, w64, x, b, m, n, k, DTYPE_F32)  # (the weights meet x in f32)


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("m,k", [(1, 512), (2, 264), (4, 512)])
def test_the_two_row_kernels_agree_bitwise(gpu, dtype, m, k):
    """Rows in flight whole, and two pieces at a time: each lane adds the same products in the same order."""
    n = 2049  # rows of one piece a lane: the one kernel up to 2048 of them, the other from there on
    w, _, x, b = make(m, n, k, dtype)
    run = lambda rows: sa.linear(sa.LinearWeight(w[:rows * k].copy(), dtype, rows, k), x, b[:rows].copy(),
                                 StreamingLinearConfig(m, k, rows)).reshape(m, rows)
    assert_bitwise(run(n)[:, :n - 1], run(n - 1), "2049 rows against 2048")
