"""The SpMM kernel for narrow rows of B, which stages a long segment a workgroup: every width it takes and the ones beside them,
rows around what a lane group, a wave and a segment take, segments of one row and of empty rows only, sizes at which its segments
are shortest, one round, longest and full turns, and a B that 32-bit offsets do not span.  Products of small integers, whose sums
are exact in both types and in any order, against integer sums."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


def _check(lens, k, ncols, dtype, planned, pad=0, beta=0.5):
    rng = np.random.default_rng(len(lens) + ncols)
    m, rp = len(lens), np.r_[0, np.cumsum(lens)].astype(np.int32)
    ldb, ldc = ncols + pad, ncols + 2 * pad
    col, val = rng.integers(0, k, rp[-1]).astype(np.int32), rng.integers(-3, 4, rp[-1]).astype(dtype)
    B, C0 = rng.integers(-3, 4, (k, ldb)).astype(dtype), 2 * rng.integers(-3, 4, (m, ldc)).astype(dtype)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, B, C0)]
    plan = capi.Plan(True, capi.SPMM_MERGE, val.dtype, m, k, col.size, d[0], ncols=ncols, col=d[1], val=d[2]) if planned else None
    capi.spmm(*d, ncols, 2.0, beta, alg=capi.SPMM_MERGE, plan=plan, ldb=ldb, ldc=ldc, k=k)
    # one column at a time: cumulative sums of integers, exact in float64
    ref = C0.copy()
    for c in range(ncols):
        s = np.r_[0.0, np.cumsum(val.astype(np.float64) * B[col, c])]
        ref[:, c] = 2.0 * (s[rp[1:]] - s[rp[:-1]]) + beta * C0[:, c]
    assert np.array_equal(d[4].cpu().numpy(), ref), (ncols, planned, pad)
    if plan is not None:
        plan.destroy()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ncols", [1, 2, 3, 4, 5, 7, 8, 9, 16])
@pytest.mark.parametrize("planned", [False, True])
def test_rows_of_every_kind(dtype, ncols, planned):
    rng = np.random.default_rng(1)
    edges = [0, 1, 7, 8, 9, 63, 64, 65, 255, 256, 257, 511, 671, 672, 673, 1343, 1344, 1345, 2687, 2688, 2689, 6001]
    lens = np.r_[rng.integers(0, 30, 700), np.repeat(edges, 2), np.zeros(4000, int), rng.permutation(edges), 3000, 1]
    _check(lens, 500, ncols, dtype, planned, pad=3, beta=0.0)
    _check(rng.integers(5, 40, 900), 333, ncols, dtype, planned)


@pytest.mark.parametrize("dtype,ncols", [(np.float32, 2), (np.float32, 16), (np.float64, 2), (np.float64, 8)])
@pytest.mark.parametrize("m,per,ragged", [(1, 9, 0), (300, 20, 0), (40000, 20, 5), (61000, 20, 0), (205000, 20, 0), (200000, 20, 9), (21000, 192, 0),
                                          (3000, 1344, 0), (1500, 1440, 0), (600, 2000, 700)])
def test_segment_sizes(dtype, ncols, m, per, ragged):
    lens = np.full(m, per) + (np.random.default_rng(m).integers(-ragged, ragged + 1, m) if ragged else 0)
    for planned in (False, True):
        _check(lens, 4000, ncols, dtype, planned)


def test_wide_b():
    k, ldb, m = 9, 1 << 27, 3000  # 4.8 GB of B
    gen = torch.Generator(device="cuda").manual_seed(5)
    B = torch.zeros((k, ldb), device="cuda")
    B[:, :8] = torch.randint(-3, 4, (k, 8), device="cuda", generator=gen).float()
    rp = (torch.arange(m + 1, device="cuda") * 12).to(torch.int32)
    col = torch.randint(0, k, (m * 12,), device="cuda", generator=gen, dtype=torch.int32)
    val = torch.randint(-3, 4, (m * 12,), device="cuda", generator=gen).float()
    C = torch.zeros((m, 8), device="cuda")
    capi.spmm(rp, col, val, B, C, 8, 1.0, 0.0, ldb=ldb, ldc=8, k=k)
    ref = (val[:, None] * B[:, :8][col.long()]).reshape(m, 12, 8).sum(1)
    assert torch.equal(C, ref)


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("k", [None, 1])
def test_view_of_a_matrix_beyond_4_gb(planned, k):
    """Eight of 64 columns of 20 M rows, 5.1 GB from the first row to the last, by calls that do not say how many rows there are
    and by calls that say too few."""
    rows, m = 20_000_000, 30000
    gen = torch.Generator(device="cuda").manual_seed(6)
    B = torch.empty((rows, 64), device="cuda")[:, :8]
    B.copy_(torch.randint(-3, 4, B.shape, device="cuda", generator=gen, dtype=torch.int8))
    rp = (torch.arange(m + 1, device="cuda") * 12).to(torch.int32)
    col = torch.randint(0, rows, (m * 12,), device="cuda", generator=gen, dtype=torch.int32)
    col[-1] = rows - 1
    val = torch.randint(-3, 4, (m * 12,), device="cuda", generator=gen).float()
    C = torch.zeros((m, 8), device="cuda")
    plan = capi.Plan(True, capi.SPMM_DEFAULT, val.dtype, m, rows, col.numel(), rp, ncols=8, col=col, val=val) if planned else None
    capi.spmm(rp, col, val, B, C, 8, 1.0, 0.0, plan=plan, ldb=64, ldc=8, k=k)
    ref = (val[:, None] * B[col.long()]).reshape(m, 12, 8).sum(1)
    assert torch.equal(C, ref)
    if plan is not None:
        plan.destroy()


@pytest.mark.parametrize("ncols", [4, 8])
@pytest.mark.parametrize("rows", [(1 << 24) - 1, 1 << 24])
def test_offsets_up_to_4_gb(rows, ncols):
    """Rows of 256 bytes up to 2^32 - 256 bytes, whose offsets a planned call holds in 32 bits where a lane takes 4 columns, and one
    row more; the same with 8 columns, which it multiplies out."""
    m = 30000
    gen = torch.Generator(device="cuda").manual_seed(7)
    B = torch.empty((rows, 64), device="cuda")
    B[:, -ncols:].copy_(torch.randint(-3, 4, (rows, ncols), device="cuda", generator=gen, dtype=torch.int8))
    rp = (torch.arange(m + 1, device="cuda") * 12).to(torch.int32)
    col = torch.randint(0, rows, (m * 12,), device="cuda", generator=gen, dtype=torch.int32)
    col[::7] = rows - 1
    val = torch.randint(-3, 4, (m * 12,), device="cuda", generator=gen).float()
    C = torch.zeros((m, ncols), device="cuda")
    plan = capi.Plan(True, capi.SPMM_DEFAULT, val.dtype, m, rows, col.numel(), rp, ncols=ncols, col=col, val=val)
    capi.spmm(rp, col, val, B[:, -ncols:], C, ncols, 1.0, 0.0, plan=plan, ldb=64, ldc=ncols)
    assert plan.info("shared_segments") == 1
    assert torch.equal(C, (val[:, None] * B[:, -ncols:][col.long()]).reshape(m, 12, ncols).sum(1))
    plan.destroy()


@pytest.mark.parametrize("dtype,ncols", [(np.float32, n) for n in (33, 57, 65, 101, 129, 257, 300)] + [(np.float64, n) for n in (17, 33, 65, 129, 301)])
@pytest.mark.parametrize("planned", [False, True])
def test_wide_rows_of_b(dtype, ncols, planned):
    """Every number of lanes a row and one or more tiles of them; rows around what a group, a wave and a segment take, each added to
    C once; the fewest items a segment holds, the most of one round, and more than a round (where only scattered columns come here,
    so that these run the merge kernel)."""
    rng = np.random.default_rng(ncols)
    edges = [0, 1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 639, 640, 641, 1279, 1281]
    _check(np.r_[rng.integers(0, 12, 300), edges, np.zeros(900, int), rng.permutation(edges), 1500, 1], 500, ncols, dtype, planned, pad=3)
    _check([3], 5, ncols, dtype, planned, beta=0.0)
    turns = -(-ncols * np.dtype(dtype).itemsize // 512)
    for work in (768 * 128 + 5, 768 * 640 - 9, 768 * 640 + 4000):
        per = 11
        _check(np.r_[np.full(work // turns // (per + 1), per), 700], 3000, ncols, dtype, planned)


@pytest.mark.parametrize("dtype,ncols", [(torch.float32, n) for n in (65, 129, 257, 300)] + [(torch.float64, n) for n in (33, 65, 129, 301)])
@pytest.mark.parametrize("rows", [3000, 60000])
def test_scattered_columns(dtype, ncols, rows):
    """DEFAULT's plan for columns that lie all over B: tiles of up to 1 KB, 32 and 64 lanes a row of B, where several rounds of
    workgroups (60000 rows) come here for the columns alone; rows around what a wave and a segment take, cut ones among them."""
    k, gen = 200000, torch.Generator(device="cuda").manual_seed(ncols)
    edges = torch.tensor([0, 1, 7, 8, 9, 63, 64, 65, 127, 128, 129, 511, 512, 513, 639, 640, 641, 1281, 5000])
    lens = torch.cat([torch.randint(4, 15, (rows,), generator=torch.Generator().manual_seed(rows)), edges, torch.zeros(700, dtype=torch.int64), edges])
    rp = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(torch.int32).cuda()
    m, nnz = lens.numel(), int(lens.sum())
    col = torch.randint(0, k, (nnz,), device="cuda", generator=gen, dtype=torch.int32)
    draw = lambda *shape: torch.randint(-3, 4, shape, device="cuda", generator=gen).to(dtype)
    val, B, C = draw(nnz), draw(k, ncols), 2 * draw(m, ncols)
    row = torch.repeat_interleave(torch.arange(m, device="cuda"), lens.cuda())
    ref = 2 * torch.zeros_like(C).index_add_(0, row, val[:, None] * B[col.long()]) + 0.5 * C
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, k, nnz, rp, ncols=ncols, col=col, val=val)
    capi.spmm(rp, col, val, B, C, ncols, 2.0, 0.5, plan=plan)
    assert torch.equal(C, ref)
    several = (m + nnz) * -(-ncols * val.element_size() // 512) > 768 * 640
    assert plan.info("shared_segments") == 1 and several == (rows == 60000)
    plan.destroy()


@pytest.mark.parametrize("dtype,ncols", [(np.float32, n) for n in (9, 12, 17, 25, 32)] + [(np.float64, n) for n in (5, 6, 10, 13, 16)])
@pytest.mark.parametrize("planned", [False, True])
def test_rows_of_b_between_narrow_and_wide(dtype, ncols, planned):
    """The fewest items a segment holds, the most, and more than one round of segments; rows that are cut and rows that are not."""
    for work in (768 * 256 - 3, 768 * 256 + 900, 768 * 1344 - 9, 768 * 1344 + 4000):
        _check(np.full(work // 15, 14), 3000, ncols, dtype, planned)
    _check(np.r_[np.full(3000, 11), 5000, np.zeros(700, int), 255, 256, 257, 511, 512, 513], 700, ncols, dtype, planned, pad=1)


def _microseconds(per, ncols, dtype, elements=6_000_000):
    """Of a planned multiply with even rows of `per` elements within 2 * per of the diagonal, the least of several."""
    m, k = elements // per, 100000
    gen = torch.Generator(device="cuda").manual_seed(per)
    rp = (torch.arange(m + 1, device="cuda") * per).to(torch.int32)
    low = (torch.arange(m, device="cuda") * k // m - 2 * per).clamp(0, k - 4 * per)
    col = (low[:, None] + 4 * torch.arange(per, device="cuda")[None, :]).reshape(-1).to(torch.int32)
    val = torch.rand(m * per, device="cuda", generator=gen, dtype=dtype)
    B, C = torch.rand((k, ncols), device="cuda", generator=gen, dtype=dtype), torch.empty((m, ncols), device="cuda", dtype=dtype)
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, k, m * per, rp, ncols=ncols, col=col, val=val)
    ws = torch.empty(max(plan.workspace_bytes, 256), dtype=torch.uint8, device="cuda")
    best = 1e9
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            capi.spmm(rp, col, val, B, C, ncols, 1.0, 0.0, plan=plan, workspace=ws)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 100)
    plan.destroy()
    return best


@pytest.mark.parametrize("dtype,ncols", [(torch.float64, 2), (torch.float64, 5), (torch.float32, 3), (torch.float32, 11)])
@pytest.mark.parametrize("per", [90, 180])
def test_as_many_elements_in_rows_that_a_wave_takes(dtype, ncols, per):
    """Little longer than in rows that a lane group takes: the waves of a workgroup share them.  Where the wave that dealt rows out
    took the long ones of its own, seven of eight had nothing to do and it took 2.3 to 4.3 times as long.  The bound: up to 64 lane
    groups of a wave have four rows of B in flight each, 256 places for 180 elements, 1.42, and then add up over six shuffles."""
    assert _microseconds(per, ncols, dtype) < 1.8 * _microseconds(60, ncols, dtype)


@pytest.mark.parametrize("dtype,ncols", [(torch.float32, 2), (torch.float32, 6), (torch.float32, 16), (torch.float64, 2), (torch.float64, 8)])
@pytest.mark.parametrize("per,shared", [(3, 0), (4, 1)])
def test_short_rows_of_large_matrices(dtype, ncols, per, shared):
    """Rows of 3 stay with one wave a segment, which is 5 % faster for them on average; rows of 4 go to whole workgroups."""
    m = 4_000_000 // (per + 1) + 1
    rp = (torch.arange(m + 1, device="cuda") * per).to(torch.int32)
    gen = torch.Generator(device="cuda").manual_seed(per)
    col = torch.randint(0, m, (m * per,), device="cuda", generator=gen, dtype=torch.int32)
    val = torch.randint(-3, 4, (m * per,), device="cuda", generator=gen).to(dtype)
    B = torch.randint(-3, 4, (m, ncols), device="cuda", generator=gen).to(dtype)
    C = torch.zeros((m, ncols), device="cuda", dtype=dtype)
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, m, m * per, rp, ncols=ncols, col=col, val=val)
    capi.spmm(rp, col, val, B, C, ncols, 1.0, 0.0, plan=plan)
    assert torch.equal(C, (val[:, None] * B[col.long()]).reshape(m, per, ncols).sum(1))
    assert plan.info("shared_segments") == shared
    plan.destroy()


@pytest.mark.parametrize("ncols,dtype,groups", [(8, np.float64, 16), (16, np.float32, 16), (4, np.float64, 32), (2, np.float64, 64)])
@pytest.mark.parametrize("per", [5, 10, 15, 19, 20, 21])
def test_even_rows_fill_whole_turns(ncols, dtype, groups, per):
    """Segments of several rounds end with a turn of all lane groups that is full or more than half full."""
    m = 8_000_000 // (per + 1)
    rp = (torch.arange(m + 1, device="cuda") * per).to(torch.int32)
    gen = torch.Generator(device="cuda").manual_seed(per)
    t = torch.float64 if dtype == np.float64 else torch.float32
    col = ((torch.arange(m, device="cuda")[:, None] + torch.arange(per, device="cuda")) % m).reshape(-1).to(torch.int32)
    val = torch.randint(-3, 4, (m * per,), device="cuda", generator=gen).to(t)
    B = torch.randint(-3, 4, (m, ncols), device="cuda", generator=gen).to(t)
    C = torch.zeros((m, ncols), device="cuda", dtype=t)
    plan = capi.Plan(True, capi.SPMM_MERGE, t, m, m, m * per, rp, ncols=ncols, col=col, val=val)
    capi.spmm(rp, col, val, B, C, ncols, 1.0, 0.0, alg=capi.SPMM_MERGE, plan=plan)
    assert torch.equal(C, (val[:, None] * B[col.long()]).reshape(m, per, ncols).sum(1))
    turn = groups * 8 * (per + 1)
    rest = plan.info("segment_items") % turn
    assert plan.info("shared_segments") == 1 and (rest == 0 or 2 * rest > min(turn, 2688)), (plan.info("segment_items"), turn)
    plan.destroy()


@pytest.mark.parametrize("dtype,ncols", [(torch.float64, 3), (torch.float32, 8)])
@pytest.mark.parametrize("per,rows,rounds", [(9, 38904, 1), (8, 62000, 1), (16, 121000, 1), (16, 125000, 2), (9, 412000, 2)])
def test_segments_fill_whole_rounds(dtype, ncols, per, rows, rounds):
    """One round of workgroups or two, three a compute unit, whatever whole turns of their lane groups take of even rows."""
    rp = (torch.arange(rows + 1, device="cuda") * per).to(torch.int32)
    gen = torch.Generator(device="cuda").manual_seed(per)
    col = torch.randint(0, rows, (rows * per,), device="cuda", generator=gen, dtype=torch.int32)
    val = torch.randint(-3, 4, (rows * per,), device="cuda", generator=gen).to(dtype)
    B = torch.randint(-3, 4, (rows, ncols), device="cuda", generator=gen).to(dtype)
    C = torch.zeros((rows, ncols), device="cuda", dtype=dtype)
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, rows, rows, rows * per, rp, ncols=ncols, col=col, val=val)
    ref = (val[:, None] * B[col.long()]).reshape(rows, per, ncols).sum(1)
    for p in (plan, None):
        C.fill_(-1)
        capi.spmm(rp, col, val, B, C, ncols, 1.0, 0.0, plan=p)
        assert torch.equal(C, ref)
    total = rows * (per + 1)
    assert plan.info("shared_segments") == 1
    filled = max(672, -(-total // (768 * rounds)))
    assert 15 * filled <= 16 * plan.info("segment_items") <= 16 * filled  # without a last turn of a sixteenth
    plan.destroy()


@pytest.mark.parametrize("ncols,dtype", [(2, np.float64), (4, np.float64), (8, np.float32), (4, np.float32)])
@pytest.mark.parametrize("rows,per", [(60000, 16), (62000, 16), (130000, 16), (30000, 45)])
def test_long_rows_and_no_plan_around_one_round(ncols, dtype, rows, per):
    """Rows that are cut, with a plan and without: one round of workgroups goes to whole workgroups, more to the waves unless rows of B
    hold 4 columns fp32 at most."""
    lens = np.full(rows, per)
    lens[::997] = 4000
    total = rows + int(lens.sum())
    for planned in (True, False):
        _check(lens, 5000, ncols, dtype, planned)
    rp = torch.from_numpy(np.r_[0, np.cumsum(lens)].astype(np.int32)).cuda()
    col = torch.zeros(int(lens.sum()), dtype=torch.int32, device="cuda")
    val = torch.zeros(col.numel(), dtype=torch.float64 if dtype == np.float64 else torch.float32, device="cuda")
    plan = capi.Plan(True, capi.SPMM_MERGE, val.dtype, rows, 5000, col.numel(), rp, ncols=ncols, col=col, val=val)
    assert plan.info("shared_segments") == int(total <= 768 * 1344 or (dtype == np.float32 and ncols <= 4))
    assert plan.info("shared_segments") or plan.info("segment_items") <= 512
    plan.destroy()
