"""The two-column streaming kernel (opy_tv_wide, TVBatch(multi_kernel="auto")
on one-channel FP32 batches): strips of 128 - 2K columns, two per lane.  Its
iterates are those of K single launches bit for bit."""
import numpy as np
import pytest

from test_gpu_tv_batch import rects

pytestmark = pytest.mark.gpu

# widths at and around one strip (128), two strips of the extended layout
# (128 + 128 - 2K) and of the plain one, odd ones, one column; heights of one
# row, below and above the units' rows and the 2K steps before the first store
SHAPES = [(130, 200), (1, 100), (97, 1), (5, 128), (40, 129), (17, 113), (23, 241), (64, 2), (150, 127), (30, 371),
          (200, 256)]


def _run(multi, kernel, steps, rows, monkeypatch, shapes=SHAPES, iters=24):
    from opymize_amd.solvers import tv
    monkeypatch.setattr(tv, "WIDE_ROWS", (rows,))
    imgs = [rects(H, W, 3 + i) for i, (H, W) in enumerate(shapes)]
    lams = [1.0 + 1.7 * i for i in range(len(shapes))]
    data = ["l1" if i % 3 == 1 else "l2" for i in range(len(shapes))]
    bat = tv.TVBatch(imgs, lams, data, tvw=[1.0 + 0.1 * i for i in range(len(shapes))], tile=(64, 4), multi=multi,
                     multi_kernel=kernel)
    res = bat.solve(steps=steps, step_bound=0.124, max_iters=2 * iters, block_iters=iters, tol=1e-30)
    if multi > 1:
        assert bat._use_wide(bat._cfg(steps)) == (kernel == "auto") and bat.wrows == rows
    return bat.solution(), [r["gap"] for r in res]


@pytest.mark.parametrize("steps", ["accel", "const"])
@pytest.mark.parametrize("multi,rows", [(2, 8), (3, 40), (4, 8), (5, 256), (6, 32), (7, 8), (8, 8), (8, 40), (8, 256),
                                        (2, 1), (4, 3), (8, 1), (8, 2)])
def test_wide_equals_single_launches(gpu, monkeypatch, multi, rows, steps):
    """Two blocks of a whole number of launches and a remainder of single
    iterations (25 = 3 * 8 + 1), TV-L1 and TV-L2, uneven TV weights."""
    (xs, ys), gaps = _run(multi, "auto", steps, rows, monkeypatch, iters=25)
    (x1, y1), gaps1 = _run(1, "auto", steps, rows, monkeypatch, iters=25)
    for a, b in zip(xs + ys, x1 + y1):
        np.testing.assert_array_equal(a, b)
    assert gaps == gaps1


@pytest.mark.parametrize("multi,block", [(8, 6), (8, 7), (8, 13), (8, 15), (4, 7), (5, 9), (3, 5), (8, 2)])
def test_rest_of_a_block_takes_few_launches(gpu, monkeypatch, multi, block):
    """What a block leaves over of whole launches (all of it where it is
    shorter than one) runs on tiles of up to four iterations, at most one
    iteration by itself; the iterates of single launches, captured or not."""
    from opymize_amd.solvers import tv
    imgs = [rects(H, W, 3 + i) for i, (H, W) in enumerate(SHAPES)]
    data = ["l1" if i % 3 == 1 else "l2" for i in range(len(SHAPES))]
    out = []
    for m, graph in ((multi, False), (multi, True), (1, True)):
        bat = tv.TVBatch(imgs, 3.0, data, multi=m)
        names = []
        call = bat._call
        monkeypatch.setattr(bat, "_call", lambda name, *a: (names.append(name), call(name, *a))[1])
        res = bat.solve(steps="accel", step_bound=0.124, max_iters=4 * block, block_iters=block, tol=1e-30,
                        use_graph=graph)
        out.append((bat.solution(), [r["gap"] for r in res]))
        if m > 1 and not graph:
            rest = block % multi
            count = [names.count("opy_tv_" + k) for k in ("wide_f32", "multi_f32", "iter_f32")]
            assert count == [4 * (block // multi), 4 * ((rest + 2) // 4), 4 * (rest % 4 == 1)]
        if m == 8:
            assert bat._captured(bat._cfg("accel"), False, block) == (block < 8)
    for (xs, ys), gaps in out[:2]:
        for a, b in zip(xs + ys, out[2][0][0] + out[2][0][1]):
            np.testing.assert_array_equal(a, b)
        assert gaps == out[2][1]


@pytest.mark.parametrize("multi", [3, 8])
def test_wide_launch_shapes(gpu, multi):
    """A block per unit, as many as are resident at once and seven, each of
    which walks many units: the same iterates and gaps, bit for bit, after every
    number of launches a check sees."""
    from opymize_amd.solvers import tv
    imgs = [rects(H, W, 3 + i) for i, (H, W) in enumerate(SHAPES)]
    data = ["l1" if i % 3 == 1 else "l2" for i in range(len(SHAPES))]
    out = {}
    for grid in (None, 0, 7):
        bat = tv.TVBatch(imgs, 3.0, data, multi=multi, grid=grid)
        assert bat.wgrid == (grid if grid is not None else bat.wgrid)
        res = bat.solve(steps="accel", step_bound=0.124, max_iters=72, block_iters=24, tol=1e-30)
        assert bat._use_wide(bat._cfg("accel"))
        units = int(bat.wide_off.cpu()[-1])
        assert units > 100 and bat.wgrid == (-(-units // 8) * 8 if grid is None else grid)
        out[grid] = (bat.solution(), [r["gap"] for r in res])
    for g in (0, 7):
        for a, b in zip(out[None][0][0] + out[None][0][1], out[g][0][0] + out[g][0][1]):
            np.testing.assert_array_equal(a, b)
        assert out[None][1] == out[g][1]


@pytest.mark.parametrize("multi,block,graph", [(8, 130, False), (7, 130, False), (6, 64, False), (5, 68, False),
                                               (3, 130, True), (3, 130, False), (8, 72, False)])
def test_blocks_longer_than_a_step_table(gpu, multi, block, graph):
    """One table holds the steps of at most 64 iterations, in whole launches
    (63 for 7 or 3 per launch, 60 for 5): blocks that take a second and a third
    one carry the schedule on from table to table; the iterates and steps of
    single launches, bit for bit, and the same over a second solve."""
    from opymize_amd.solvers import tv
    imgs = [rects(H, W, 50 + i) for i, (H, W) in enumerate([(40, 129), (97, 1), (64, 150), (9, 300)])]
    out = []
    for m, g in ((multi, graph), (1, True)):
        bat = tv.TVBatch(imgs, [2.0, 9.0, 15.0, 19.0], ["l2", "l1", "l2", "l2"], multi=m)
        names = []
        call = bat._call
        bat._call = lambda name, *a: (names.append(name), call(name, *a))[1]
        for _ in range(2):
            bat.set_start(None, None)
            res = bat.solve(steps="accel", step_bound=0.124, step_factor=4.0, max_iters=3 * block, block_iters=block,
                            tol=1e-30, use_graph=g)
        out.append((bat.solution(), [r["gap"] for r in res], bat.steps_state()))
        if m > 1 and not g:
            per = tv.WIDE_TABLE - tv.WIDE_TABLE % m
            assert names.count("opy_tv_wide_steps") == 6 * -(-(block - block % m) // per)
            assert names.count("opy_tv_wide_f32") == 6 * (block // m)
    for a, b in zip(out[0][0][0] + out[0][0][1], out[1][0][0] + out[1][0][1]):
        np.testing.assert_array_equal(a, b)
    assert out[0][1] == out[1][1]
    for a, b in zip(out[0][2], out[1][2]):
        assert (a["tau"], a["sigma"]) == (b["tau"], b["sigma"])


def test_kernel_may_change_between_blocks(gpu, monkeypatch):
    """Fewer than 6 iterations per launch: one column per lane while the batch
    is large, two from the check on at which enough instances stopped; captured
    blocks and the iterates of single launches, bit for bit."""
    from opymize_amd.solvers import tv
    monkeypatch.setattr(tv, "WIDE_UNITS", {3: 6})
    imgs = [rects(H, W, 30 + i) for i, (H, W) in enumerate([(60, 140), (33, 250), (90, 64), (20, 300)])]
    out = []
    for multi in (3, 1):
        bat = tv.TVBatch(imgs, [2.0, 9.0, 15.0, 19.0], "l2", multi=multi)
        used = []
        res = bat.solve(steps="accel", step_bound=0.124, step_factor=4.0, max_iters=4800, block_iters=48, tol=1e-5,
                        callback=lambda b, n: used.append(b._wide_now))
        out.append(([(r["iter"], r["gap"], r["status"]) for r in res], bat.solution()))
        if multi > 1:
            assert not used[0] and True in used
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1][0] + out[0][1][1], out[1][1][0] + out[1][1][1]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("multi,side,n,wide", [(2, 1024, 14, True), (2, 1024, 16, False), (4, 512, 60, True),
                                               (4, 512, 110, False), (5, 512, 110, True), (5, 512, 210, False),
                                               (6, 512, 210, True)])
def test_large_batches_below_six_per_launch(gpu, multi, side, n, wide):
    """Which kernel a batch takes either side of WIDE_UNITS."""
    import torch
    from opymize_amd.solvers import tv
    bat = tv.TVBatch([np.zeros((side, side))] * n, 3.0, "l2", multi=multi)
    bat.solve(steps="accel", step_bound=0.124, max_iters=multi, block_iters=multi, tol=0.0)
    bat.checks.zero_()  # all running, whatever the check of a zero image says
    bat._compact(0)
    assert bat.refresh_grid() == n
    assert bat._use_wide(bat._cfg("accel")) == wide
    del bat
    torch.cuda.empty_cache()


def test_wide_units_follow_the_running_instances(gpu):
    """The device's unit prefixes against a host recount, after some
    instances stopped; rows chosen for the whole and the reduced set."""
    import torch
    from opymize_amd.solvers import tv
    imgs = [rects(H, W, 9 + i) for i, (H, W) in enumerate(SHAPES)]
    bat = tv.TVBatch(imgs, 3.0, "l2", multi=8)
    bat.solve(steps="accel", step_bound=0.124, max_iters=8, block_iters=8, tol=1e-30)
    ck = bat.checks.view(torch.int32).reshape(bat.B, -1)
    for b in (0, 4, 10):
        ck[b, 16] = 1  # status field of opy_tv_check_t: certified
    bat._compact(0)
    nrun = bat.refresh_grid()
    active = bat.active_inst.cpu().numpy()[:nrun]
    assert nrun == bat.B - 3 and not {0, 4, 10} & set(active.tolist())
    for off, strips, rows in ((bat.wide_off, tv._wide_strips(bat._W, 112), bat.wrows),
                              (bat.unit_off, bat._strips, bat.stream_rows)):
        counts = (strips * -(-bat._H // rows))[active]
        np.testing.assert_array_equal(off.cpu().numpy()[:nrun + 1], np.concatenate([[0], np.cumsum(counts)]))


def test_units_entry_points_agree(gpu):
    """opy_tv_stream_units writes the prefix that opy_tv_wide_units writes
    beside its own, for every number of iterations per launch."""
    import torch
    from opymize_amd import _hip
    from opymize_amd.solvers import tv
    P = _hip.ptr
    bat = tv.TVBatch([rects(H, W, 9 + i) for i, (H, W) in enumerate(SHAPES)], 3.0, "l2", multi=8)
    bat.solve(steps="accel", step_bound=0.124, max_iters=8, block_iters=8, tol=1e-30)
    for k in range(2, 9):
        for rows in (1, 16, 128):
            a, b, c = (torch.full((bat.B + 1,), -1, dtype=torch.int32, device="cuda") for _ in range(3))
            bat._call("opy_tv_stream_units", P(bat.insts), P(bat.active_inst), P(bat.nact), P(a), k, rows,
                      _hip.stream())
            bat._call("opy_tv_wide_units", P(bat.insts), P(bat.active_inst), P(bat.nact), k, P(b), rows, P(c), 32,
                      _hip.stream())
            counts = [tv._stream_strips(W, 64 - 2 * k) * -(-H // rows) for H, W in SHAPES]
            np.testing.assert_array_equal(a.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
            assert torch.equal(a, b)


def test_wide_graph_replays_equal_eager(gpu, monkeypatch):
    """Captured blocks (the step table among them) replayed many times against
    eager launches, on a batch that certifies instance by instance."""
    from opymize_amd.solvers import tv
    monkeypatch.setattr(tv, "CAPTURE_BELOW", 9)  # capture at 8 iterations per launch too
    imgs = [rects(H, W, 30 + i) for i, (H, W) in enumerate([(60, 140), (33, 250), (90, 64), (20, 300)])]
    out = []
    for g in (True, False):
        bat = tv.TVBatch(imgs, [2.0, 9.0, 15.0, 19.0], "l2", multi=8)
        res = bat.solve(steps="accel", step_bound=0.124, step_factor=4.0, max_iters=4800, block_iters=48, tol=1e-5,
                        use_graph=g)
        out.append(([(r["iter"], r["gap"], r["status"]) for r in res], bat.solution()))
    assert out[0][0] == out[1][0] and all(s == 1 for _, _, s in out[0][0])
    for a, b in zip(out[0][1][0] + out[0][1][1], out[1][1][0] + out[1][1][1]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("kernel", ["auto", "stream"])
@pytest.mark.parametrize("graph", [True, False])
def test_stopped_instances_keep_their_iterate_over_odd_blocks(gpu, monkeypatch, graph, kernel):
    """Three launches of 8 iterations per block: the buffers change places
    at every check, and an instance certified at one of them keeps the iterate
    that was certified, whichever buffer later blocks end in (single launches
    as the reference, bit for bit)."""
    from opymize_amd.solvers import tv
    monkeypatch.setattr(tv, "CAPTURE_BELOW", 9)
    imgs = [rects(H, W, 30 + i) for i, (H, W) in enumerate([(60, 140), (33, 250), (90, 64), (20, 300)])]
    out = []
    for multi in (8, 1):
        bat = tv.TVBatch(imgs, [2.0, 9.0, 15.0, 19.0], "l2", multi=multi, multi_kernel=kernel)
        bat.stream_min_units = 0
        mid = []
        res = bat.solve(steps="accel", step_bound=0.124, step_factor=4.0, max_iters=2400, block_iters=24, tol=1e-5,
                        use_graph=graph, callback=lambda b, n: mid.append(b.solution()[0][0]) if n <= 240 else None)
        out.append(([(r["iter"], r["gap"], r["status"]) for r in res], bat.solution(), mid))
    its = [i // 24 for i, _, s in out[0][0]]
    assert len(set(i % 2 for i in its)) == 2  # stopped in different buffers
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1][0] + out[0][1][1] + out[0][2], out[1][1][0] + out[1][1][1] + out[1][2]):
        np.testing.assert_array_equal(a, b)


def test_wide_entry_points_refuse_bad_arguments():
    """Host checks before any launch."""
    import ctypes
    from opymize_amd import _hip
    from opymize_amd.solvers import tv
    tv._bind()
    lib = _hip.load()
    assert lib.opy_tv_wide_f32(*([None] * 7), 8, 0, None, None, None, 9, 8, 8, None) == 1
    assert b"k = 9" in lib.opy_last_error()
    q = ctypes.c_void_p(64)
    args = [q, ctypes.c_void_p(128), q, ctypes.c_void_p(128), q, q, q]
    assert lib.opy_tv_wide_f32(*args, 8, 1, q, q, q, 8, 8, 8, None) == 1  # iterations 1..9 of 8
    assert b"outside the table" in lib.opy_last_error()
    c = tv.TVCfg()
    c.C, c.tw, c.rpt, c.steps, c.h0, c.h1 = 1, 64, 4, tv.STEP_MODES["precond"], 1.0, 1.0
    assert lib.opy_tv_wide_steps(q, q, q, 1, ctypes.byref(c), 8, q, None) == 1
    assert b"preconditioned" in lib.opy_last_error()
