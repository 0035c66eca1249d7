"""GPU `sum` split (ekv_rank_sum through allocate and sum_keep) bit-exact against the oracle:
the reference test's tied integer scores with weights, explicit pins, float64 scores, rows past
NumPy's 8192-value reduction run, and the view-build configuration at full size
(observe/allocation.py:55-123 and tests/test_allocation.py:170-250 of the reference)."""

import numpy as np
import pytest
import torch

import workloads
from cases import random_requests
from observe import allocation
from oracle import allocation as oa

pytestmark = pytest.mark.gpu


def same(got, want):
    return len(got) == len(want) and all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("seed", range(40))
def test_sum_with_ties_and_weights(seed):
    rng = np.random.default_rng(seed)
    reqs = []
    for _ in range(int(rng.integers(1, 9))):
        n = int(rng.integers(3, 40))
        scores = rng.integers(0, 4, size=n).astype(float)  # many equal scores, so many ties
        reqs.append(allocation.Request(scores=scores, weight=float(rng.choice([1.0, 2.0, 0.5]))))
    total = sum(len(r.scores) for r in reqs)
    must = sum(int(r.pinned_mask().sum()) for r in reqs)
    budget = int(rng.integers(must, max(total, must + 1)))
    got = allocation.allocate(reqs, budget, "sum")
    want = oa.allocate_sum([r.scores for r in reqs], [r.pinned_mask() for r in reqs], [r.weight for r in reqs], budget)
    assert same(got, want)


def test_sum_float64_scores_and_explicit_pins():
    rng = np.random.default_rng(3)
    for trial in range(60):
        scores, pinned = random_requests(rng, int(rng.integers(1, 7)), 50, ties=trial % 2 == 0)
        scores = [s.astype(np.float64) * (1 + 1e-9 * rng.random(len(s))) for s in scores]  # not float32 values
        weights = [float(rng.choice([1.0, 3.0, 0.25])) for _ in scores]
        total = sum(len(s) for s in scores)
        must = sum(int(p.sum()) for p in pinned)
        budget = int(rng.integers(must, max(total, must + 1)))
        reqs = [allocation.Request(scores=s, weight=w, pinned=p) for s, w, p in zip(scores, weights, pinned)]
        assert same(allocation.allocate(reqs, budget, "sum"), oa.allocate_sum(scores, pinned, weights, budget)), trial


def test_sum_row_totals_are_numpy_sums_bit_for_bit():
    # every ranking divides by NumPy's float64 sum of the clamped scores; a total one ulp off would
    # shift each share by about an ulp, which the keep masks rarely show, so the totals are read back
    # from the workspace (its state block, then one 24-byte statistic per row: the total first) and
    # compared bit for bit: lengths across the leaf sizes (1..128), the pairwise splits and several
    # 8192-value runs, with values over many binades so that the order of the additions shows
    rng = np.random.default_rng(21)
    lengths = [1, 2, 7, 8, 9, 15, 16, 17, 127, 128, 129, 136, 255, 256, 257, 1000, 1024, 4095, 4096,
               4097, 8191, 8192, 8193, 12288, 16385, 20000]
    width = max(lengths)
    rows = len(lengths)
    scores = np.zeros((rows, width))
    for r, n in enumerate(lengths):
        scores[r, :n] = rng.random(n) * 10.0 ** rng.integers(-12, 4, size=n)
        scores[r, : n : 5] *= -1.0  # clamped to 0
    state = allocation.sum_workspace_bytes(0) - 256
    stat = 24
    workspace = torch.zeros(allocation.sum_workspace_bytes(rows), dtype=torch.uint8, device="cuda")
    s_dev = torch.from_numpy(scores).cuda()
    b_dev = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    allocation.sum_keep(s_dev, b_dev, budget=sum(lengths) // 2, workspace=workspace)
    torch.cuda.synchronize()
    raw = workspace.cpu().numpy()
    base = (-workspace.data_ptr()) % 256 + state
    for r, n in enumerate(lengths):
        got = raw[base + r * stat: base + r * stat + 8].view(np.float64)[0]
        want = np.maximum(scores[r, :n], 0.0).sum()
        assert got.tobytes() == np.float64(want).tobytes(), (n, got, want)


def test_sum_rows_past_one_reduction_run():
    # rows of more than 8192 blocks: NumPy's total adds two runs' pairwise sums
    rng = np.random.default_rng(8)
    scores = [rng.random(n) * rng.choice([1e-3, 1.0, 7.0]) for n in (8191, 8192, 8193, 12288, 9000)]
    pinned = [oa.default_pins(len(s)) for s in scores]
    weights = [1.0, 2.0, 0.5, 1.0, 1.5]
    total = sum(len(s) for s in scores)
    for frac in (0.1, 0.5, 0.9):
        budget = int(frac * total)
        reqs = [allocation.Request(scores=s, weight=w) for s, w in zip(scores, weights)]
        assert same(allocation.allocate(reqs, budget, "sum"), oa.allocate_sum(scores, pinned, weights, budget)), frac


def test_sum_rows_wider_than_a_register_row():
    # rows past 12288 blocks and past the 14-bit block field of the narrower tie key (16384): the tie
    # passes cover 18 bits of block; integer scores force ties at the threshold across requests, and
    # NumPy's totals add several 8192-value runs
    rng = np.random.default_rng(16)
    for sizes in ((16384, 12289, 300), (16385, 32768, 5000), (40000, 17, 20000)):
        scores = [rng.integers(0, 5, size=n).astype(float) * rng.choice([1e-3, 1.0]) for n in sizes]
        scores[0][::7] = 2.0  # many equal gains
        pinned = [oa.default_pins(len(x)) for x in scores]
        weights = [1.0, 2.0, 1.0][: len(sizes)]
        total = sum(sizes)
        for frac in (0.2, 0.5):
            budget = int(frac * total)
            reqs = [allocation.Request(scores=x, weight=w) for x, w in zip(scores, weights)]
            print(f"sizes {sizes} budget {budget}", flush=True)
            assert same(allocation.allocate(reqs, budget, "sum"), oa.allocate_sum(scores, pinned, weights, budget))


def test_sum_view_build_configuration():
    # 1024 rows of U[1, 8192] blocks with Dirichlet(0.1) float32 shares: budgets 0.2 / 0.5 / 0.8
    c = workloads.config4()
    shares, blocks = c["shares"], c["blocks"]
    sizes = blocks.tolist()
    total = int(blocks.sum())
    scores = [shares[r, : sizes[r]] for r in range(len(sizes))]
    pinned = [oa.default_pins(n) for n in sizes]
    s_dev, b_dev = torch.from_numpy(shares).cuda(), torch.from_numpy(blocks).cuda()
    for frac in (0.2, 0.5, 0.8):
        budget = int(np.ceil(frac * total))
        keep, summary = allocation.sum_keep(s_dev, b_dev, budget=budget)
        got = keep.cpu().numpy()
        want = oa.allocate_sum(scores, pinned, [1.0] * len(sizes), budget)
        bad = sum(int((got[r, : sizes[r]].astype(bool) != want[r]).sum()) for r in range(len(sizes)))
        print(f"sum at {frac}: budget {budget}, kept {sum(int(w.sum()) for w in want)}, mismatched {bad}", flush=True)
        assert bad == 0 and int(summary[0]) == budget and int(summary[3]) == 0
        assert all(got[r, sizes[r]:].all() for r in range(len(sizes))), "a position past a row is kept"


def test_sum_select_ending_at_the_first_digit():
    # the free blocks are exactly the open blocks of the top bucket of the first digit (shares near 1/k
    # against shares 1e-10 times smaller, 33 binades apart): the select ends at the first pass, so the
    # keep kernel writes every block itself; a budget one block larger ends it in a later pass
    rng = np.random.default_rng(5)
    scores, pinned = [], []
    for n in (40, 300, 3000, 9000):
        big = int(rng.integers(5, n - 5))
        x = np.concatenate([1.0 + rng.random(big), 1e-10 * (1.0 + rng.random(n - big))])
        scores.append(rng.permutation(x))
        pinned.append(oa.default_pins(n))
    must = sum(int(p.sum()) for p in pinned)
    top = sum(int(((x >= 1.0) & ~p).sum()) for x, p in zip(scores, pinned))
    for budget in (must + top, must + top + 1, must + top - 1):
        reqs = [allocation.Request(scores=x) for x in scores]
        assert same(allocation.allocate(reqs, budget, "sum"), oa.allocate_sum(scores, pinned, [1.0] * 4, budget)), budget


def test_sum_more_than_65536_requests():
    # 70000 requests: the tie key's request field takes 17 bits; integer scores tie across requests
    rng = np.random.default_rng(31)
    rows, width = 70000, 6
    scores = rng.integers(0, 3, size=(rows, width)).astype(np.float64)
    sizes = rng.integers(1, width + 1, size=rows)
    pinned = [oa.default_pins(int(n)) for n in sizes]
    total = int(sizes.sum())
    s_dev = torch.from_numpy(scores).cuda()
    b_dev = torch.from_numpy(sizes.astype(np.int32)).cuda()
    must = sum(int(p.sum()) for p in pinned)
    for frac in (0.3, 0.6):
        budget = must + int(frac * (total - must))
        keep, summary = allocation.sum_keep(s_dev, b_dev, budget=budget)
        got = keep.cpu().numpy()
        want = oa.allocate_sum([scores[r, : sizes[r]] for r in range(rows)], pinned, [1.0] * rows, budget)
        bad = sum(int((got[r, : sizes[r]].astype(bool) != want[r]).sum()) for r in range(rows))
        print(f"sum over {rows} requests at {frac}: mismatched {bad}", flush=True)
        assert bad == 0 and int(summary[4]) == rows


def test_maxmin_more_than_65536_requests():
    # 70000 requests: the bisection's state in memory, its summed count and active requests packed
    rng = np.random.default_rng(32)
    rows, width = 70000, 6
    scores = rng.random((rows, width)) * rng.choice([1e-3, 1.0], size=(rows, 1))
    sizes = rng.integers(1, width + 1, size=rows)
    pinned = [oa.default_pins(int(n)) for n in sizes]
    total = int(sizes.sum())
    s_dev = torch.from_numpy(scores).cuda()
    b_dev = torch.from_numpy(sizes.astype(np.int32)).cuda()
    must = sum(int(p.sum()) for p in pinned)
    budget = must + int(0.5 * (total - must))
    keep, summary = allocation.maxmin_keep(s_dev, b_dev, budget=budget)
    got = keep.cpu().numpy()
    want = oa.allocate_maxmin([scores[r, : sizes[r]] for r in range(rows)], pinned, budget)
    bad = sum(int((got[r, : sizes[r]].astype(bool) != want[r]).sum()) for r in range(rows))
    print(f"maxmin over {rows} requests: mismatched {bad}", flush=True)
    assert bad == 0 and int(summary[4]) == rows


@pytest.mark.parametrize("rows,width", [(127, 300), (128, 512), (129, 513), (130, 2048), (131, 2049), (511, 40),
                                        (512, 512), (513, 511), (700, 513), (1025, 64), (128, 1025), (255, 1300),
                                        (256, 1792), (300, 1793), (600, 2048)])
@pytest.mark.parametrize("kind", ["shares", "ties"])
def test_sum_rows_side_by_side(rows, width, kind):
    # the passes take a row with 64, 256 or 1024 threads by the number of rows and the width: both sides of
    # each line, with lists that hold (shares) and that outgrow their room (many equal gains), pins and
    # weights, strided keeps; whole numbers, so equal to the oracle's
    rng = np.random.default_rng(700 + rows + width)
    sizes = rng.integers(0, width + 1, size=rows)
    sizes[0] = width
    scores = rng.gamma(0.1, size=(rows, width)) if kind == "shares" else rng.integers(0, 2, (rows, width)).astype(float)
    pins = rng.random((rows, width)) < 0.05
    weights = rng.uniform(0.5, 2.0, size=rows) if kind == "shares" else np.ones(rows)
    must, total = int(sum(pins[r, : sizes[r]].sum() for r in range(rows))), int(sizes.sum())
    budget = must + (total - must) // 2
    out = torch.full((rows, width + 5), 7, dtype=torch.uint8, device="cuda")
    keep, summary = allocation.sum_keep(
        torch.from_numpy(scores).cuda(), torch.from_numpy(sizes.astype(np.int32)).cuda(), budget=budget,
        weights=torch.from_numpy(weights).cuda(), pinned=torch.from_numpy(pins.astype(np.uint8)).cuda(),
        out=out[:, :width])
    want = oa.allocate_sum([scores[r, : sizes[r]] for r in range(rows)], [pins[r, : sizes[r]] for r in range(rows)],
                           list(weights), budget)
    got = keep.cpu().numpy()
    for r in range(rows):
        assert np.array_equal(got[r, : sizes[r]].astype(bool), want[r]), (r, sizes[r])
        assert (got[r, sizes[r]:] == 1).all()
    assert (out[:, width:] == 7).all() and summary.tolist()[:4] == [budget, total, must, 0]


@pytest.mark.parametrize("rows_past,per_cu,width", [(44, 1, 3000), (1, 1, 2049), (100, 4, 1500)])
def test_sum_lists_have_room_for_every_row_of_their_workgroup(rows_past, per_cu, width):
    # row counts that leave some workgroups of the passes a row more than the others (one or four rows side
    # by side): 900 blocks a row in one first digit are within the 1024 pairs that a row brings to its
    # workgroup's list, so every one of them is found in the workspace (a list without room for a
    # workgroup's second row makes each later pass read the rows again)
    rows = torch.cuda.get_device_properties(0).multi_processor_count * per_cu + rows_past
    rng = np.random.default_rng(rows + width)
    scores = np.zeros((rows, width))
    for r in range(rows):
        listed = rng.choice(np.arange(1, width - 1), size=900, replace=False)
        scores[r, listed] = rng.uniform(1.0, 1.5, size=900)  # shares of 900 such: within a quarter of 1 / 1125
    need = allocation.sum_workspace_bytes(rows)
    workspace = torch.zeros(need, dtype=torch.uint8, device="cuda")
    budget = 2 * rows + 450 * rows
    keep, summary = allocation.sum_keep(
        torch.from_numpy(scores).cuda(), torch.full((rows,), width, dtype=torch.int32, device="cuda"), budget=budget,
        workspace=workspace)
    assert summary.tolist()[:4] == [budget, rows * width, 2 * rows, 0] and int(keep.sum()) == budget
    words = workspace[(-workspace.data_ptr()) % 8:]
    words = words[: words.numel() // 8 * 8].view(torch.int64).cpu().numpy()
    row, block = np.nonzero(scores)
    tie_keys = (block.astype(np.int64) << 16) | (65535 - row)
    assert np.isin(tie_keys, words).all()


def test_sum_summary_flags_a_budget_below_the_pins():
    scores = torch.ones(2, 5, dtype=torch.float64, device="cuda")
    blocks = torch.tensor([5, 5], dtype=torch.int32, device="cuda")
    keep, summary = allocation.sum_keep(scores, blocks, budget=3)  # 4 pinned blocks
    assert int(summary[3]) == 1 and int(summary[2]) == 4
    with pytest.raises(ValueError):
        allocation.allocate([allocation.Request(scores=np.ones(5))] * 2, 3, "sum")


# ---- maxmin ----------------------------------------------------------------------------------

def test_maxmin_running_totals_are_numpy_cumsums_bit_for_bit():
    # the running totals of each request's open shares sorted by share (np.cumsum) are read back from
    # the workspace (the last rows x width float64 array before its 256-byte tail) and compared bit for
    # bit: shares with full mantissas, whose sums round to ties about half the time while a share is
    # within a binade of the total; coarse integer scores (many equal shares); exact binary fractions;
    # shares across 300 decades; zero plateaus; lengths on both sides of the 1024-value chunks; a NaN
    # score (every share NaN) and a +inf score (zero shares, then one NaN, which sorts last)
    rng = np.random.default_rng(33)
    lengths = [1, 2, 3, 17, 1023, 1024, 1025, 1026, 2047, 2049, 3000, 4096, 5000, 8191, 8192, 8192,
               6000, 7000, 8000, 300, 9000, 12288, 2500, 3100]
    width = max(lengths)
    rows = len(lengths)
    scores = np.zeros((rows, width))
    for r, n in enumerate(lengths):
        kind = r % 6
        if kind == 0:
            x = rng.dirichlet(np.full(n, 0.1))
        elif kind == 1:
            x = rng.integers(1, 9, size=n).astype(np.float64)
        elif kind == 2:
            x = np.full(n, 0.25)
        elif kind == 3:
            x = rng.random(n) * 10.0 ** rng.uniform(-300, 0, size=n)
        elif kind == 4:
            x = rng.random(n)
            x[rng.random(n) < 0.7] = 0.0
        else:
            x = rng.dirichlet(np.full(n, 10.0))
        if r == len(lengths) - 2:
            x = rng.random(n)
            x[n // 3] = np.nan
        elif r == len(lengths) - 1:
            x = rng.random(n)
            x[n // 2] = np.inf
        scores[r, :n] = x
    need = allocation.maxmin_workspace_bytes(rows, width)
    workspace = torch.zeros(need, dtype=torch.uint8, device="cuda")
    s_dev = torch.from_numpy(scores).cuda()
    b_dev = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    total = sum(lengths)
    must = sum(min(n, 2) for n in lengths)
    allocation.maxmin_keep(s_dev, b_dev, budget=must + (total - must) // 2, workspace=workspace)
    torch.cuda.synchronize()
    raw = workspace.cpu().numpy()
    cells = rows * width * 8
    prefix = (-workspace.data_ptr()) % 256 + need - 256 - (cells + 255) // 256 * 256
    for r, n in enumerate(lengths):
        with np.errstate(invalid="ignore"):
            sh = oa.shares(scores[r, :n])  # inf / inf is NaN
        open_sh = sh[~oa.default_pins(n)]
        nan = np.isnan(open_sh)
        want = np.cumsum(np.concatenate([np.sort(open_sh[~nan])[::-1], open_sh[nan]]))
        got = raw[prefix + r * width * 8: prefix + (r * width + len(want)) * 8].view(np.float64)
        assert np.array_equal(np.isnan(got), np.isnan(want)), (n, r)
        fin = ~np.isnan(want)
        assert got[fin].tobytes() == want[fin].tobytes(), (n, r % 6, int(np.argmax(got != want)))


@pytest.mark.parametrize("width", [300, 512, 513, 1024, 1025, 3000, 4096, 4097, 8192])
@pytest.mark.parametrize("masked", [False, True])
def test_maxmin_rows_of_one_workgroup(width, masked):
    # requests of at most 8192 blocks go from scores to running totals in one workgroup: ranks from
    # buckets of the shares' leading bits, or a radix sort when too many unequal shares crowd in one or
    # the shares span more than 512 binades; totals in workgroup-wide windows.  Lengths at the
    # edges of a thread's blocks, a wave and the row; the totals bit for bit np.cumsum's, the keep the
    # oracle's (NaN and inf rows: the totals only)
    rng = np.random.default_rng(900 + width + masked)
    lengths = [n for n in (1, 2, 3, 63, 64, 65, 255, 257, 511, 600, 1023, 2047, 2049, 4095, 5000, 8191, width - 1,
                           width, width, width, width, width, width, width, width // 2) if n <= width]
    rows = len(lengths)
    scores, pins = [], []
    for r, n in enumerate(lengths):
        kind = r % 8
        if kind == 0:
            x = rng.dirichlet(np.full(n, 0.1)).astype(np.float32).astype(np.float64)
        elif kind == 1:
            x = rng.integers(1, 9, size=n).astype(np.float64)
        elif kind == 2:
            x = rng.random(n) * 10.0 ** rng.uniform(-300, 0, size=n)
        elif kind == 3:
            x = rng.random(n)
            x[rng.random(n) < 0.7] = 0.0
        elif kind == 4:
            x = rng.dirichlet(np.full(n, 10.0))
        elif kind == 5:
            x = 1.0 + rng.random(n) * 2.0 ** -30  # shares that differ in their low bits only
        elif kind == 6:
            x = np.repeat(rng.dirichlet(np.full(n, 0.3)), 2)[:n]
        else:
            x = np.where(rng.random(n) < 0.5, rng.random(n), 0.0)
            x[: n // 100] = 0.0
        scores.append(x)
        if masked:
            pin = rng.random(n) < rng.choice([0.0, 0.02, 0.5])
            pin[0] = True
            pins.append(pin)
        else:
            pins.append(oa.default_pins(n))
    finite = rows
    for special in (np.nan, np.inf):
        x = rng.random(width)
        x[width // 3] = special
        scores.append(x)
        lengths = lengths + [width]
        pins.append(oa.default_pins(width))
    for count, check_keep in ((finite, True), (finite + 2, False)):
        grid = np.zeros((count, width))
        mask = np.zeros((count, width), bool)
        for r in range(count):
            grid[r, : lengths[r]] = scores[r]
            mask[r, : lengths[r]] = pins[r]
        need = allocation.maxmin_workspace_bytes(count, width)
        workspace = torch.zeros(need, dtype=torch.uint8, device="cuda")
        total = sum(lengths[:count])
        must = sum(int(p.sum()) for p in pins[:count])
        budget = must + (total - must) // 2
        keep, summary = allocation.maxmin_keep(
            torch.from_numpy(grid).cuda(), torch.tensor(lengths[:count], dtype=torch.int32, device="cuda"),
            budget=budget, pinned=torch.from_numpy(mask.astype(np.uint8)).cuda() if masked else None,
            workspace=workspace)
        assert summary.tolist()[:4] == [budget, total, must, 0]
        raw = workspace.cpu().numpy()
        cells = count * width * 8
        prefix = (-workspace.data_ptr()) % 256 + need - 256 - (cells + 255) // 256 * 256
        for r in range(count):
            with np.errstate(invalid="ignore"):
                sh = oa.shares(scores[r])  # inf / inf is NaN
            open_sh = sh[~pins[r]]
            nan = np.isnan(open_sh)
            want = np.cumsum(np.concatenate([np.sort(open_sh[~nan])[::-1], open_sh[nan]]))
            got = raw[prefix + r * width * 8: prefix + (r * width + len(want)) * 8].view(np.float64)
            assert np.array_equal(np.isnan(got), np.isnan(want)), (lengths[r], r)
            fin = ~np.isnan(want)
            assert got[fin].tobytes() == want[fin].tobytes(), (lengths[r], r % 8)
        if check_keep:
            want = oa.allocate_maxmin(scores[:count], pins[:count], budget)
            got = keep.cpu().numpy().astype(bool)
            for r in range(count):
                assert np.array_equal(got[r, : lengths[r]], want[r]), (lengths[r], r % 8)


@pytest.mark.parametrize("seed", range(40))
def test_maxmin_random_requests(seed):
    rng = np.random.default_rng(seed)
    scores, pinned = random_requests(rng, int(rng.integers(1, 9)), 40)
    total = sum(len(s) for s in scores)
    must = sum(int(p.sum()) for p in pinned)
    budget = int(rng.integers(must, max(total, must + 1)))
    reqs = [allocation.Request(scores=s, pinned=p) for s, p in zip(scores, pinned)]
    assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget))


def test_maxmin_identical_requests_and_edges():
    # identical requests reach the level together: the leftover goes one block each by index
    rng = np.random.default_rng(4)
    s = rng.dirichlet(np.full(30, 0.3))
    scores = [s.copy() for _ in range(12)]
    pinned = [oa.default_pins(30) for _ in scores]
    must = sum(int(p.sum()) for p in pinned)
    for budget in (must, must + 1, must + 7, must + 100, 360 - 1, 360):
        reqs = [allocation.Request(scores=x) for x in scores]
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), budget
    with pytest.raises(ValueError):
        allocation.allocate([allocation.Request(scores=np.ones(5))] * 2, 3, "maxmin")


@pytest.mark.parametrize("rows", [12, 1500, 3000])
def test_maxmin_leftover_over_plateaus_and_ties(rows):
    # a large leftover: requests whose remaining shares are zero (a plateau the level bisection stops
    # below) take every block they have left at one level; equal shares, shares too small to move the
    # level and distinct ones mixed across requests; 1500 and 3000 requests put 2 and 4 on a thread
    rng = np.random.default_rng(rows)
    scores = []
    for r in range(rows):
        n = int(rng.integers(3, 60))
        kind = r % 4
        if kind == 0:
            x = np.zeros(n)
            x[0] = 1.0  # one block carries everything: the rest are a zero plateau
        elif kind == 1:
            x = np.ones(n)  # equal shares
        elif kind == 2:
            x = np.full(n, 1e-30)
            x[0] = 1.0  # shares below the level's last bit once the first block is kept
        else:
            x = rng.random(n)
        scores.append(x)
    pinned = [oa.default_pins(len(x)) for x in scores]
    total = sum(len(x) for x in scores)
    must = sum(int(q.sum()) for q in pinned)
    for frac in (0.3, 0.6, 0.95):
        budget = max(must, int(frac * total))
        reqs = [allocation.Request(scores=x) for x in scores]
        print(f"{rows} requests, budget {budget} of {total}", flush=True)
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


@pytest.mark.parametrize("sizes", [(12289, 300, 5000), (20000, 16384, 17, 9000), (65535, 40000, 12288),
                                   (65536, 100000, 7), (262144, 70000)])
def test_maxmin_rows_wider_than_a_sort_in_lds(sizes):
    # requests past 12288 blocks sort in global memory and search their running
    # totals in memory; ties (integer scores), explicit pins and a zero tail
    rng = np.random.default_rng(sum(sizes))
    scores = [rng.integers(0, 6, size=n).astype(float) * rng.choice([1e-3, 1.0]) for n in sizes]
    scores[0][-(len(scores[0]) // 5):] = 0.0
    pinned = [oa.default_pins(len(x)) for x in scores]
    pinned[1] = pinned[1].copy()
    pinned[1][:: 97] = True
    total = sum(sizes)
    must = sum(int(q.sum()) for q in pinned)
    for frac in (0.2, 0.55, 0.9):
        budget = max(must, int(frac * total))
        reqs = [allocation.Request(scores=x, pinned=q) for x, q in zip(scores, pinned)]
        print(f"sizes {sizes}, budget {budget}", flush=True)
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


def test_maxmin_float64_scores_zero_rows_and_long_rows():
    rng = np.random.default_rng(6)
    scores = [rng.random(n) * (1 + 1e-9 * rng.random(n)) for n in (8191, 8193, 12288, 50)]
    scores.append(np.zeros(40))  # no evidence: equal shares
    scores.append(np.array([0.0, -1.0, 2.0, np.float64(1e-300)]))
    pinned = [oa.default_pins(len(s)) for s in scores]
    pinned[3] = rng.random(50) < 0.3  # explicit pins
    total = sum(len(s) for s in scores)
    for frac in (0.05, 0.3, 0.7, 0.95):
        budget = max(int(frac * total), sum(int(p.sum()) for p in pinned))
        reqs = [allocation.Request(scores=s, pinned=p) for s, p in zip(scores, pinned)]
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


@pytest.mark.parametrize("spread", [2.0 ** -40, 2.0 ** -30, 2.0 ** -26])
def test_maxmin_shares_that_differ_only_in_low_bits(spread):
    # shares a few float64 ulps apart (1 + k * spread, a handful of distinct values per row), next to rows
    # whose shares differ high up: the row kernel's bins span the row's own shares, so each value has a
    # bucket (the radix sort's second sort: test_maxmin_rows_past_8192_blocks_sorted_again and
    # test_maxmin_equal_shares_keep_block_order)
    rng = np.random.default_rng(int(-np.log2(spread)))
    scores = []
    for n in (8192, 4096, 3000, 1024, 700, 64):
        s = 0.5 * (1.0 + rng.integers(0, 7, size=n) * spread)
        if n == 3000:
            s = rng.random(n)  # no close neighbours
        scores.append(s)
    pinned = [oa.default_pins(len(s)) for s in scores]
    total = sum(len(s) for s in scores)
    for frac in (0.1, 0.5, 0.9):
        budget = max(int(frac * total), sum(int(q.sum()) for q in pinned))
        reqs = [allocation.Request(scores=s, pinned=q) for s, q in zip(scores, pinned)]
        print(f"spread {spread}, budget {budget}", flush=True)
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


def test_maxmin_ties_in_rows_sorted_in_lds():
    # each request's blocks are ranked in LDS by share desc, equal shares in block order: rows full of
    # exactly equal shares must keep the stable order the reference's argsort gives
    rng = np.random.default_rng(9)
    scores = [np.round(rng.random(n) * 8) / 8 for n in (8192, 4097, 1000, 64)]  # 9 distinct values
    scores.append(np.full(300, 0.25))
    scores.append(np.zeros(40))
    pinned = [oa.default_pins(len(s)) for s in scores]
    pinned[2] = rng.random(1000) < 0.2
    total = sum(len(s) for s in scores)
    for frac in (0.1, 0.4, 0.6, 0.9):
        budget = max(int(frac * total), sum(int(p.sum()) for p in pinned))
        reqs = [allocation.Request(scores=s, pinned=p) for s, p in zip(scores, pinned)]
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


def test_maxmin_view_build_configuration():
    c = workloads.config4()
    shares, blocks = c["shares"], c["blocks"]
    sizes = blocks.tolist()
    total = int(blocks.sum())
    scores = [shares[r, : sizes[r]] for r in range(len(sizes))]
    pinned = [oa.default_pins(n) for n in sizes]
    s_dev, b_dev = torch.from_numpy(shares).cuda(), torch.from_numpy(blocks).cuda()
    for frac in (0.2, 0.5, 0.8):
        budget = int(np.ceil(frac * total))
        keep, summary = allocation.maxmin_keep(s_dev, b_dev, budget=budget)
        got = keep.cpu().numpy()
        want = oa.allocate_maxmin(scores, pinned, budget)
        bad = sum(int((got[r, : sizes[r]].astype(bool) != want[r]).sum()) for r in range(len(sizes)))
        print(f"maxmin at {frac}: budget {budget}, kept {sum(int(w.sum()) for w in want)}, mismatched {bad}",
              flush=True)
        assert bad == 0 and int(summary[3]) == 0


@pytest.mark.parametrize("rows", [1500, 3000, 6000, 8192, 8193, 20000])
def test_maxmin_many_requests(rows):
    # past 1024 requests each bisection thread carries 2, 4 or 8 of them; past 8192 the bisection
    # keeps every request's state in the workspace
    rng = np.random.default_rng(rows)
    sizes = rng.integers(1, 30, size=rows)
    scores = [rng.random(int(n)) for n in sizes]
    scores[5] = np.zeros(int(sizes[5]))
    pinned = [oa.default_pins(int(n)) for n in sizes]
    total, must = int(sizes.sum()), sum(int(p.sum()) for p in pinned)
    for frac in (0.3, 0.75):
        budget = max(int(frac * total), must)
        reqs = [allocation.Request(scores=s, pinned=p) for s, p in zip(scores, pinned)]
        assert same(allocation.allocate(reqs, budget, "maxmin"), oa.allocate_maxmin(scores, pinned, budget)), frac


def maxmin_order_and_totals(scores, pins, width, masked):
    """A call's requests' open blocks in sorted order and their running totals, read from the workspace
    (rows of at most 12288 blocks), beside NumPy's; the keep is checked against the oracle."""
    rows, lengths = len(scores), [len(x) for x in scores]
    grid, mask = np.zeros((rows, width)), np.zeros((rows, width), np.uint8)
    for r in range(rows):
        grid[r, : lengths[r]], mask[r, : lengths[r]] = scores[r], pins[r]
    need = allocation.maxmin_workspace_bytes(rows, width)
    workspace = torch.zeros(need, dtype=torch.uint8, device="cuda")
    must = sum(int(p.sum()) for p in pins)
    budget = must + (sum(lengths) - must) // 2
    keep, summary = allocation.maxmin_keep(
        torch.from_numpy(grid).cuda(), torch.tensor(lengths, dtype=torch.int32, device="cuda"), budget=budget,
        pinned=torch.from_numpy(mask).cuda() if masked else None, workspace=workspace)
    assert summary.tolist()[:4] == [budget, sum(lengths), must, 0]
    want_keep, keep = oa.allocate_maxmin(scores, pins, budget), keep.cpu().numpy().astype(bool)
    raw = workspace.cpu().numpy()
    prefix = (-workspace.data_ptr()) % 256 + need - 256 - (rows * width * 8 + 255) // 256 * 256
    vals = prefix - (rows * width * 4 + 255) // 256 * 256
    for r in range(rows):
        share = oa.shares(scores[r])
        blocks = np.flatnonzero(~pins[r])
        blocks = blocks[np.argsort(-share[blocks], kind="stable")]
        totals = np.cumsum(share[blocks])
        got_order = raw[vals + r * width * 4: vals + (r * width + len(blocks)) * 4].view(np.int32)
        got = raw[prefix + r * width * 8: prefix + (r * width + len(blocks)) * 8].view(np.float64)
        assert np.array_equal(got_order, blocks), (r, lengths[r], int(np.argmax(got_order != blocks)))
        assert got.tobytes() == totals.tobytes(), (r, lengths[r], int(np.argmax(got != totals)))
        assert np.array_equal(keep[r, : lengths[r]], want_keep[r]), (r, lengths[r])


def share_keys(scores, pins):
    """The order-preserving keys of a request's open shares (not negative): larger share, larger key."""
    share = oa.shares(scores)[~pins]
    return share.view(np.uint64) | np.uint64(1 << 63)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("kind", [2.0 ** -40, 2.0 ** -30, 2.0 ** -26, "ties"])
def test_maxmin_rows_past_8192_blocks_sorted_again(kind, masked):
    # a call with rows of 8193 to 12288 blocks takes the LDS radix sort for every request, with 1, 2, 4, 8 or
    # 12 keys a thread; shares that agree in their top 40 bits out of order below are sorted again
    # (spreads of a few float64 ulps), equal ones keep block order
    rng = np.random.default_rng(42 if kind == "ties" else int(-np.log2(kind)))
    scores, pins = [], []
    for n in (12288, 9000, 8193, 8192, 5000, 4096, 2049, 2048, 1025, 1024, 700, 64):
        scores.append(np.round(rng.random(n) * 8) / 8 if kind == "ties" else 0.5 * (1.0 + rng.integers(0, 7, n) * kind))
        pins.append(oa.default_pins(n) if not masked else rng.random(n) < 0.05)
        top, low = share_keys(scores[-1], pins[-1]) >> 24, share_keys(scores[-1], pins[-1]) & 0xffffff
        order = np.argsort(top, kind="stable")[::-1]  # runs of equal top bits, each from its last block
        again = (top[order][1:] == top[order][:-1]) & (low[order][1:] < low[order][:-1])
        assert again.any() == (kind != "ties" and kind < 2.0 ** -28), n
    maxmin_order_and_totals(scores, pins, 12288, masked)


def bucket_case(scores, pins):
    """How the row kernel's ranks take a request: the bits that every bucket has to fix (2 and more: the
    shares span more than 512 binades and take the radix sort)."""
    keys = share_keys(scores, pins)
    keys = keys[keys > np.uint64(1 << 63)]
    span = int(keys.max() - keys.min())
    cut = max(0, (span | 1).bit_length() - 9)
    cut += (span >> cut) >= 511
    return max(0, cut + 13 - 64)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("width", [512, 1024, 4096, 8192])
def test_maxmin_shares_over_many_binades(width, masked):
    # shares over 200 to 600 binades: below 256 a bucket's word holds all that the bucket leaves open;
    # from there to 511 every bucket has to fix one bit more; past that the request takes the radix
    # sort.  Whole rows with several blocks a coarse bin, the order read from the workspace (the totals
    # stop changing after the first binades)
    rng = np.random.default_rng(width + masked)
    scores, pins, cases = [], [], []
    for binades in (200, 254, 258, 300, 400, 500, 508, 513, 600):
        x = np.ldexp(1.0 + rng.random(width), rng.integers(-binades, 1, width))
        x[[width // 3, width // 2]] = [1.0, np.ldexp(1.0, -binades)]  # the whole range, unpinned
        pin = rng.random(width) < 0.05 if masked else oa.default_pins(width)
        pin[[width // 3, width // 2]] = False
        scores.append(x)
        pins.append(pin)
        cases.append(bucket_case(x, pin))
    assert cases == [0, 0, 1, 1, 1, 1, 1, 2, 2]
    maxmin_order_and_totals(scores, pins, width, masked)


def window_ties(share, threads):
    """The scan windows of a request's sorted open shares, as the row kernel takes them with this many
    threads: (ties in the window, whether it is a wide one) for each."""
    totals = np.cumsum(share)
    windows, pos, n = [], 0, len(share)
    alone, wide = True, False
    t = -0.0
    while pos < n:
        if alone or not t > 0.0:
            pos = min(pos + 64, n)
            t, alone = totals[pos - 1], False
            continue
        u = np.spacing(t)
        asked = min(n - pos, (8 if wide else 2) * threads)
        y = share[pos: pos + asked] / u  # exact: u is a power of two
        tie = y - np.floor(y) == 0.5
        before = np.concatenate([[t], totals[pos: pos + asked - 1]])
        under = y < 2.0 ** 53 - before / u
        windows.append((int(tie.sum()), wide))
        if tie.sum() > 64:
            asked = min(n - pos, 2 * threads)
            stop = ~under[:asked] | tie[:asked]
            taken = int(np.argmax(stop)) if stop.any() else asked
            alone = taken < asked
        else:
            taken = int(np.argmax(~under)) if not under.all() else asked
            alone, wide = taken < 64, taken == asked
        if taken:
            t = totals[pos + taken - 1]
        pos += taken
        if pos < n and taken < asked and not alone:
            t = totals[pos]
            pos += 1
    return windows


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("width,threads", [(512, 256), (1024, 256), (4096, 512), (8192, 512)])
def test_maxmin_totals_with_many_ties_in_a_window(width, threads, masked):
    # a tie (a share that is an odd multiple of half the total's last bit) is resolved in place up to 64 a
    # window; more of them end the window at the first.  Shares in units of 2^-54 on a total in [1/2, 1),
    # whose last bit is 2^-53: odd ones tie.  The first and last block, pinned, hold the rest of the
    # request, set so that NumPy's total is 1 and the shares are the scores.
    scores, pins, seen = [], [], []

    def row(big, small):
        x = np.concatenate([[0.0, big], np.asarray(small, float) * 2.0 ** -54, [0.25]])
        x[0] = 0.75 - big - np.sum(x[2:-1])
        while np.sum(x) != 1.0:
            x[0] += 1.0 - np.sum(x)
        pin = np.zeros(len(x), bool)
        pin[[0, -1]] = True
        scores.append(x)
        pins.append(pin)
        assert np.array_equal(oa.shares(x), x)
        seen.append(window_ties(np.sort(x[1:-1])[::-1], threads))

    rng = np.random.default_rng(width + masked)
    m = width - 3  # small shares of a whole row
    row(0.6, np.full(m, 3))  # every value ties
    row(0.6, rng.choice([2, 3, 4, 5, 6, 7], m))
    for count in (64, 65):  # that many ties in the first window
        row(0.6, np.concatenate([np.full(100, 4), np.full(count, 3), np.full(m - 100 - count, 2)]))
        assert seen[-1][0] == (count, False)
    if width > 3 * threads:  # a whole window without ties, then a wide one with many, 64 and 65
        first = 64 + 2 * threads
        for count in (64, 65, m - first):
            row(0.6, np.concatenate([np.full(first, 4), np.full(count, 3), np.full(m - first - count, 2)]))
            assert any(w and (ties == count or 65 < ties < count) for ties, w in seen[-1])
    row(0.5 - 3 * 150 * 2.0 ** -54, np.full(m, 3))  # the total enters [1/2, 1) after 150 of them
    row(0.6, np.full(m // 2, 7))
    assert any(ties > 64 for ties, _ in seen[0]) and any(ties > 64 for ties, _ in seen[1])
    assert any(ties > 64 for ties, _ in seen[-2])
    maxmin_order_and_totals(scores, pins, width, masked)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("width", [512, 1024, 4096, 8192])
def test_maxmin_equal_shares_keep_block_order(width, masked):
    # more than 64 blocks in one of the ranks' buckets: of one share they are put in block order from a
    # bitmap; up to 128 of several shares are ranked by comparing, more send the request to the radix
    # sort and its second sort, on equal top bits (with each number of keys a thread).  Group sizes around both limits, one group, as many groups as fit (short and whole rows), in
    # random block order; the order read from the workspace
    rng = np.random.default_rng(width + masked)
    scores, pins = [], []

    def row(values):
        x = rng.permutation(np.asarray(values, float))
        scores.append(x)
        pin = rng.random(len(x)) < 0.03 if masked else oa.default_pins(len(x))
        if masked and len(x) < width:
            pin[:] = False  # the groups whole, and no pins at all
        pins.append(pin)

    for n in sorted({width, width - 1, width // 2 + 1}):
        row(np.full(n, 0.3))
        for size in (63, 64, 65, 66, 128, 129, 130, 131, 300):
            row(1.0 + np.arange(n) // size)
            row(np.where(np.arange(n) % 3, 2.0 ** -(1.0 + np.arange(n) // size % 40), 0.0))
    # one far share widens the bins, so that neighbouring float64 values share a bucket
    for size in (60, 64, 65, 100, 128, 129, 200, *sorted({min(n, width - 2) for n in (900, 1800, 3500, 8190)})):
        crowd = 1.0 + rng.integers(0, 3, size) * 2.0 ** -52
        row(np.concatenate([crowd, [1e-30, 1e-30], np.full(min(width - size - 2, 150), 2.0)]))
    row(np.concatenate([np.full(64, 1.0), [1.0 + 2.0 ** -52], [1e-30, 1e-30]]))
    row(np.concatenate([np.full(200, 1.0), [1.0 + 2.0 ** -52], [1e-30, 1e-30]]))
    maxmin_order_and_totals(scores, pins, width, masked)


@pytest.mark.parametrize("width", [512, 1024, 4096, 8192])
def test_maxmin_nan_shares_keep_block_order(width):
    # a NaN score makes every share of its request NaN: equal, in block order.  An infinite one leaves
    # zeros, which come before the NaN share of its own block
    rows, far = 4, 5
    grid = np.random.default_rng(width).random((rows, width))
    lengths = [width, width - 1, 3, width]
    grid[:3, 1] = np.nan
    grid[3, far] = np.inf
    need = allocation.maxmin_workspace_bytes(rows, width)
    workspace = torch.zeros(need, dtype=torch.uint8, device="cuda")
    allocation.maxmin_keep(torch.from_numpy(grid).cuda(), torch.tensor(lengths, dtype=torch.int32, device="cuda"),
                           budget=sum(lengths) // 2, workspace=workspace)
    raw = workspace.cpu().numpy()
    vals = (-workspace.data_ptr()) % 256 + need - 256 - (rows * width * 8 + 255) // 256 * 256 \
        - (rows * width * 4 + 255) // 256 * 256
    for r, n in enumerate(lengths):
        want = np.arange(1, n - 1)
        if r == 3:
            want = np.concatenate([want[want != far], [far]])
        got = raw[vals + r * width * 4: vals + (r * width + n - 2) * 4].view(np.int32)
        assert np.array_equal(got, want), r
