"""GPU parity of the TW mask producers (twprune, whose calls are tw_prune_tiled_wise_1d_late and its
kin; the entry points that take masks from the start in test_entry_points_with_masks_from_the_start)
against the CPU oracle and the golden vectors of the reference's prune_algo.py.

Masks are integer results: the bar is bit-exact.  The oracle computes with NumPy itself
(np.linalg.norm, np.percentile), so these tests also check that the HIP kernels repeat
NumPy's float32 summation order and percentile arithmetic."""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden", "prune_vectors.npz")


@pytest.fixture(scope="module")
def twprune(tw):
    from tilesparsity_amd import twprune as m
    return m


@pytest.fixture(scope="module")
def po():
    from oracle import tw_prune_oracle
    return tw_prune_oracle


def parse_sparsity(text):
    return int(text) if text.lstrip("-").isdigit() else float(text)


def test_golden_vectors(twprune):
    z = np.load(GOLD)
    meta = json.loads(bytes(z["meta"]).decode())
    for case in meta["cases"]:
        name, g = case["name"], case["granularity"]
        weights = [z["%s/w%d" % (name, i)] for i in range(len(case["shapes"]))]
        scores = twprune.img2col_forward(weights)
        for sp in case["sparsities"]:
            print("case", name, sp, flush=True)
            got = {"tiled_wise_1d": twprune.tiled_wise_1d(scores, parse_sparsity(sp), g),
                   "tiled_wise_2d": twprune.tiled_wise_2d(scores, parse_sparsity(sp), g)}
            for fn, masks in got.items():
                for i, m in enumerate(masks):
                    want = np.unpackbits(z["%s/%s/%s/m%d" % (name, fn, sp, i)])[:m.size]
                    assert np.array_equal(m.ravel(), want.astype(bool)), (name, fn, sp, i)


def test_norms_are_numpys_bits(twprune, po):
    rng = np.random.default_rng(20)
    for K, N, g in ((37, 300, 8), (300, 1000, 8), (64, 520, 128), (16, 1500, 700), (5, 7, 3)):
        x = rng.standard_normal((K, N)).astype(np.float32)
        table = po.tiles_every_g_columns(N, g)
        print("norms", K, N, g, flush=True)
        assert np.array_equal(twprune.tile_row_norms(x, table).view(np.uint32),
                              po.tile_row_norms(x, table).view(np.uint32))
        keep = rng.random(N) < 0.6
        want = po.tile_row_norms(x * keep[None, :], table)
        assert np.array_equal(twprune.tile_row_norms(x, table, keep).view(np.uint32), want.view(np.uint32))
        assert np.array_equal(twprune.col_norms(x).view(np.uint32), po.col_norms(x).view(np.uint32))


def test_percentile_is_numpys_bits(twprune):
    rng = np.random.default_rng(19)
    for n in (1, 2, 3, 10, 101, 1000, 37500, 300001):
        for quant in (0, 64):
            v = rng.random(n).astype(np.float32)
            if quant:
                v = (np.round(v * quant) / quant).astype(np.float32)
            for q in (0, 0.1, 25, 33.3, 50, 66.6, 75.0, 99.9, 100, np.float64(50.0), np.float64(87.3)):
                want = np.percentile(v, q)
                got = twprune.percentile(v, q)
                assert got.dtype == want.dtype and got.tobytes() == want.tobytes(), (n, quant, q, got, want)


SHAPES = [
    [(64, 256), (128, 384)],
    [(100, 130), (33, 500), (257, 64)],          # ragged last tiles
    [(300, 1000)],
    [(3, 3, 16, 48), (48, 72)],                  # conv + dense
]


@pytest.mark.parametrize("shapes", SHAPES)
@pytest.mark.parametrize("g", [8, 32, 128, 200])
@pytest.mark.parametrize("sparsity", [50, 75.0, 87.5, np.float64(60.0)])
def test_1d_matches_oracle(twprune, po, shapes, g, sparsity):
    rng = np.random.default_rng(abs(hash((str(shapes), g, float(sparsity)))) % 2 ** 31)
    scores = twprune.img2col_forward([rng.standard_normal(s).astype(np.float32) for s in shapes])
    print("1d", shapes, g, repr(sparsity), flush=True)
    want, thr, _ = po.tiled_wise_1d(scores, sparsity, g)
    got = twprune.tiled_wise_1d(scores, sparsity, g)
    assert np.float64(thr) == twprune.tiled_wise_1d.last_threshold
    for w, m in zip(want, got):
        assert np.array_equal(w, m)


@pytest.mark.parametrize("shapes", SHAPES)
@pytest.mark.parametrize("g", [8, 32, 128])
@pytest.mark.parametrize("sparsity,transform", [(50, True), (75.0, True), (60, False),
                                                (np.float64(80.0), False)])
def test_2d_matches_oracle(twprune, po, shapes, g, sparsity, transform):
    rng = np.random.default_rng(abs(hash((str(shapes), g, float(sparsity), transform))) % 2 ** 31)
    scores = twprune.img2col_forward([rng.standard_normal(s).astype(np.float32) for s in shapes])
    print("2d", shapes, g, repr(sparsity), transform, flush=True)
    want, thrs, tables, _ = po.tiled_wise_2d(scores, sparsity, g, transform=transform)
    got, got_tables = twprune.tiled_wise_2d(scores, sparsity, g, transform=transform, return_tiles=True)
    assert (np.float64(thrs[0]), np.float64(thrs[1])) == twprune.tiled_wise_2d.last_thresholds
    for w, m in zip(want, got):
        assert np.array_equal(w, m)
    assert got_tables == tables


@pytest.mark.parametrize("widths, g", [
    ([64, 65, 1, 63, 128, 4097], 1),             # tiles that end at every kept column, groups of one column
    ([140000, 7], 100),                          # more groups of 64 columns than are taken at a time, one layer across the line
    ([200] * 700, 33),                           # more of them over many layers
    ([40, 3] * 600, 5),                          # more layers than are taken at a time
    ([12288], 128), ([12289], 5000),             # columns kept in LDS, and one too many
])
def test_2d_groups_of_columns(twprune, po, widths, g):
    """The step between the stages of the 2-D producer takes the columns of all layers in groups of 64."""
    rng = np.random.default_rng(sum(widths) + g)
    scores = [np.abs(rng.standard_normal((3, n))).astype(np.float32) for n in widths]
    print("2d groups", len(widths), sum(widths), g, flush=True)
    want, _, tables, _ = po.tiled_wise_2d(scores, 60, g)
    got, got_tables = twprune.tiled_wise_2d(scores, 60, g, return_tiles=True)
    for a, b, t, u in zip(want, got, tables, got_tables):
        assert np.array_equal(a, b)
        assert [tuple(x) for x in t] == [tuple(x) for x in u]


def test_ties_and_extremes(twprune, po):
    rng = np.random.default_rng(21)
    # scores on a coarse grid: many rows share a norm, some tie with the threshold
    scores = [(np.round(rng.standard_normal((96, 128)) * 2) / 2).astype(np.float32) for _ in range(2)]
    scores = twprune.img2col_forward(scores)
    for sp in (0, 100, 50, 33.3, np.float64(66.6)):
        for g in (16, 64):
            w1, _, _ = po.tiled_wise_1d(scores, sp, g)
            g1 = twprune.tiled_wise_1d(scores, sp, g)
            w2 = po.tiled_wise_2d(scores, sp, g)[0]
            g2 = twprune.tiled_wise_2d(scores, sp, g)
            for a, b in zip(w1 + w2, g1 + g2):
                assert np.array_equal(a, b), (sp, g)
    # a constant layer: the threshold equals every norm, nothing is kept
    ones = [np.ones((8, 8), np.float32)]
    assert not twprune.tiled_wise_1d(ones, 50, 4)[0].any()


def test_wide_tiles_use_the_recursive_sum(twprune, po):
    rng = np.random.default_rng(22)
    scores = [np.abs(rng.standard_normal((40, 1500))).astype(np.float32)]
    for g in (129, 256, 700, 1500):
        want, _, _ = po.tiled_wise_1d(scores, 70, g)
        got = twprune.tiled_wise_1d(scores, 70, g)
        assert np.array_equal(want[0], got[0]), g


@pytest.mark.parametrize("shapes, g", [
    ([(33, 7 + 5 * i) for i in range(70)], 16),       # more layers than a wave's lanes, rows off 16 bytes
    ([(40, 5000), (31, 260)], 4500),                  # sums of many blocks; a remainder of rows
    ([(520, 13000)], 128),                            # more columns than the column stage keeps in LDS
])
def test_layer_and_tile_table_edges(twprune, po, shapes, g):
    rng = np.random.default_rng(25)
    scores = twprune.img2col_forward([rng.standard_normal(s).astype(np.float32) for s in shapes])
    for a, b in zip(po.tiled_wise_1d(scores, 60, g)[0], twprune.tiled_wise_1d(scores, 60, g)):
        assert np.array_equal(a, b)
    want = po.tiled_wise_2d(scores, 60, g)[0]
    for a, b in zip(want, twprune.tiled_wise_2d(scores, 60, g)):
        assert np.array_equal(a, b)


def test_masks_feed_plans(tw, twprune, po, oracle):
    """1-D masks go through tw_plan_from_mask, 2-D masks through tw_plan_from_mask_tiles with
    the kept-column tile table; the plans hold the lists the oracle derives from the mask."""
    rng = np.random.default_rng(23)
    K, N, G = 192, 320, 64
    W = rng.standard_normal((K, N)).astype(np.float32)
    scores = twprune.img2col_forward([W])
    m1 = twprune.tiled_wise_1d(scores, 75, G)[0]
    with tw.Plan.from_mask(m1, G, "f16", W) as plan:
        ex, _ = plan.export(with_weight=False)
        want = po.plan_tiles_from_mask(m1, po.tiles_every_g_columns(N, G))
        for t, wt in zip(ex, want):
            assert t["kept_k"].tolist() == wt["kept_k"] and t["kept_n"].tolist() == wt["kept_n"]
    m2, tables = twprune.tiled_wise_2d(scores, 75, G, return_tiles=True)
    with tw.Plan.from_mask_tiles(m2[0], tables[0], "f16", W) as plan:
        ex, _ = plan.export(with_weight=False)
        want = po.plan_tiles_from_mask(m2[0], tables[0])
        assert [(t["col0"], t["width"]) for t in ex] == tables[0]
        for t, wt in zip(ex, want):
            assert t["kept_k"].tolist() == wt["kept_k"] and t["kept_n"].tolist() == wt["kept_n"]
        # and the GEMM on that plan is the masked dense product
        A = rng.standard_normal((64, K)).astype(np.float32)
        from tests.test_gpu_gemm import run_gemm
        C, _ = run_gemm(tw, oracle, plan, A, "f16", N, pruned=1)
        ref = oracle.quantize(A, "f16").astype(np.float64) @ (oracle.quantize(W, "f16") * m2[0]).astype(np.float64)
        assert oracle.rel_error(C, ref) <= 1e-2


def test_granularity_pruning_matches_oracle(twprune, po):
    rng = np.random.default_rng(24)
    for K, N, g in ((64, 128, 16), (768, 768, 64), (300, 512, 128), (5, 8, 2)):
        s = np.abs(rng.standard_normal((K, N))).astype(np.float32)
        for sp in (50, 75.0, 90, np.float64(33.3), 0, 100):
            print("granularity", K, N, g, repr(sp), flush=True)
            assert np.array_equal(twprune.granularity_pruning(s, sp, g), po.granularity_pruning(s, sp, g))
    # ties inside a tile
    s = (np.round(np.abs(rng.standard_normal((96, 64))) * 2) / 2).astype(np.float32)
    assert np.array_equal(twprune.granularity_pruning(s, 60, 8), po.granularity_pruning(s, 60, 8))


@pytest.mark.parametrize("K", [1, 255, 1024, 1025, 8192, 8193])   # around the sizes where the selection changes form
@pytest.mark.parametrize("values", ["normal", "ties"])
def test_granularity_pruning_long_tiles(twprune, po, K, values):
    rng = np.random.default_rng(K)
    s = np.abs(rng.standard_normal((K, 6))).astype(np.float32)
    if values == "ties":
        s = (np.round(s * 2) / 2).astype(np.float32)
    for sp in (75, np.float64(33.3), 0, 100):
        assert np.array_equal(twprune.granularity_pruning(s, sp, 2), po.granularity_pruning(s, sp, 2)), sp


def test_granularity_pruning_of_single_columns_stays_small(twprune, po):
    """Tiles of one column: the memory of a call is a small multiple of its scores' (1 MB here), not tens of
    kilobytes a tile."""
    import torch
    rng = np.random.default_rng(26)
    s = np.abs(rng.standard_normal((16, 16384))).astype(np.float32)
    twprune.granularity_pruning(s[:, :64], 75, 1)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = twprune.granularity_pruning(s, 75, 1)
    assert free - torch.cuda.mem_get_info()[0] < 100 << 20
    assert np.array_equal(got, po.granularity_pruning(s, 75, 1))


def test_device_masks_have_storage_of_their_own(twprune):
    """return_device=True: a mask that is kept (or saved) keeps its own bytes alive and no other layer's."""
    import torch
    scores = [torch.rand(s, device="cuda") for s in ((64, 96), (33, 7), (128, 40))]
    calls = [lambda: twprune.tiled_wise_1d(scores, 60, 16, return_device=True),
             lambda: twprune.tiled_wise_2d(scores, 60, 16, return_device=True),
             lambda: twprune.tiled_wise_1d_mix(scores, 60, 16, return_device=True),
             lambda: twprune.tiled_wise_2d_mix(scores, 60, 16, return_device=True)]
    for call in calls:
        masks = call()
        assert [tuple(m.shape) for m in masks] == [tuple(s.shape) for s in scores]
        assert all(m.untyped_storage().nbytes() == m.numel() for m in masks)


def test_error_paths(tw, twprune):
    with pytest.raises(tw.TwError):
        twprune.tiled_wise_1d([np.ones((4, 4), np.float32)], 150, 2)
    with pytest.raises(tw.TwError):
        twprune.tiled_wise_1d([np.ones((4, 4), np.float32)], 50, 0)
    with pytest.raises(tw.TwError):
        twprune.granularity_pruning(np.ones((4, 6), np.float32), 50, 4)
    with pytest.raises(tw.TwError):
        tw.Plan.from_mask_tiles(np.ones((4, 8), np.uint8), [(0, 4), (5, 3)], "f16", np.ones((4, 8), np.float32))


@pytest.mark.parametrize("n_layers", [1, 128, 129])
def test_masks_of_many_layers_made_during_the_call(twprune, po, n_layers):
    """As many layers as a launch takes addresses of masks, and one more (whose addresses go to the table)."""
    rng = np.random.default_rng(n_layers)
    scores = twprune.img2col_forward([rng.standard_normal((int(rng.integers(3, 40)), int(rng.integers(3, 50)))).astype(np.float32)
                                      for _ in range(n_layers)])
    for fn in ("tiled_wise_1d", "tiled_wise_2d", "tiled_wise_1d_mix"):
        want = getattr(po, fn)(scores, 60, 16)
        want = want[0] if fn != "tiled_wise_1d_mix" else want
        got = getattr(twprune, fn)(scores, 60, 16)
        assert len(got) == n_layers and all(np.array_equal(w, g) for w, g in zip(want, got)), fn


@pytest.mark.parametrize("n_layers", [1, 20, 21, 40, 41])
def test_tables_in_the_arguments_of_the_norms(twprune, po, n_layers):
    """As many layers as go to the device with the launch that reads the scores (40, and 20 where a second stage's table goes along),
    and one more; fewer workgroups than clear the counters and more; the calls before and after it with other tables."""
    rng = np.random.default_rng(n_layers + 7)
    for rows in (8, 200):
        scores = twprune.img2col_forward([rng.standard_normal((int(rng.integers(3, rows)), 4 * int(rng.integers(1, 20)))).astype(np.float32)
                                          for _ in range(n_layers)])
        for g in (16, 12):
            for fn in ("tiled_wise_1d", "tiled_wise_1d_mix", "tiled_wise_1d"):
                want = getattr(po, fn)(scores, 60, g)
                want = want[0] if fn != "tiled_wise_1d_mix" else want
                got = getattr(twprune, fn)(scores, 60, g)
                assert len(got) == n_layers and all(np.array_equal(w, x) for w, x in zip(want, got)), (fn, rows, g)


@pytest.mark.parametrize("fn", ["tiled_wise_1d", "tiled_wise_2d", "tiled_wise_1d_mix"])
def test_masks_that_cannot_be_made_end_the_call(tw, twprune, monkeypatch, fn):
    """An exception while the masks are made comes out of the producer, and the next call is as ever."""
    rng = np.random.default_rng(3)
    scores = [rng.random((64, 96)).astype(np.float32)]
    want = getattr(twprune, fn)(scores, 50, 32)

    def fails(self):
        raise MemoryError("no masks")
    with monkeypatch.context() as m:
        m.setattr(twprune._DeviceLayers, "make_masks", fails)
        with pytest.raises(MemoryError):
            getattr(twprune, fn)(scores, 50, 32)
    assert all(np.array_equal(a, b) for a, b in zip(want, getattr(twprune, fn)(scores, 50, 32)))


@pytest.mark.parametrize("fn", ["tiled_wise_1d", "tiled_wise_2d", "tiled_wise_1d_mix"])
@pytest.mark.parametrize("n_layers", [3, 129])
def test_nothing_waits_for_a_call_that_makes_its_masks(tw, twprune, po, monkeypatch, fn, n_layers):
    """While the masks are made, the library gives back its memory, another thread's producer call comes to an end,
    and so do one of this thread and, within that, one more (more calls than there are kept buffers for): every
    call's masks are the oracle's, and so are those of the next ones."""
    import threading
    rng = np.random.default_rng(n_layers)
    scores = [rng.random((int(rng.integers(3, 90)), int(rng.integers(16, 200)))).astype(np.float32) for _ in range(n_layers)]
    want = getattr(po, fn)(scores, 60, 16)
    want = want[0] if fn != "tiled_wise_1d_mix" else want
    make, depth, results = twprune._DeviceLayers.make_masks, threading.local(), []

    def call():
        results.append(getattr(twprune, fn)(scores, 60, 16))

    def busy(self):
        at = getattr(depth, "at", 0)
        depth.at = at + 1
        print("masks", fn, n_layers, "call", at, flush=True)
        tw.release_memory()
        if at == 0:
            other = threading.Thread(target=plain)
            other.start()
            other.join(60)
            assert not other.is_alive()
        if at < 2:
            call()
        tw.release_memory()
        depth.at = at
        return make(self)

    def plain():
        depth.at = 2  # (its masks are made without further calls)
        call()
    with monkeypatch.context() as m:
        m.setattr(twprune._DeviceLayers, "make_masks", busy)
        call()
    call()
    call()
    assert len(results) == 6
    for got in results:
        assert all(np.array_equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("fn", ["tiled_wise_1d", "tiled_wise_2d", "tiled_wise_1d_mix"])
def test_calls_of_several_threads(tw, twprune, po, fn):
    """Threads in producer calls side by side, the library's memory given back now and then."""
    import threading
    rng = np.random.default_rng(8)
    jobs = [[rng.random((int(rng.integers(3, 300)), int(rng.integers(16, 400)))).astype(np.float32) for _ in range(n)] for n in (1, 3, 2, 5)]
    wants = [getattr(po, fn)(s, 60, 16) for s in jobs]
    wants = [w if fn == "tiled_wise_1d_mix" else w[0] for w in wants]
    wrong = []

    def work(i):
        try:
            for r in range(20):
                got = getattr(twprune, fn)(jobs[i], 60, 16)
                assert all(np.array_equal(a, b) for a, b in zip(wants[i], got))
                if r % 7 == i:
                    tw.release_memory()
        except BaseException as e:
            wrong.append((i, e))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(90)
    assert not wrong and not any(t.is_alive() for t in threads)


@pytest.mark.parametrize("n_layers", [3, 129])
def test_entry_points_with_masks_from_the_start(tw, twprune, n_layers):
    """tw_prune_tiled_wise_1d, _2d and _1d_mix as a C program calls them: the masks and thresholds of the calls that
    ask for their masks; a mask that is NULL, there or when it has been asked for, and a `ready` that has none
    are errors, and the next call is as ever."""
    import ctypes
    import torch
    rng = np.random.default_rng(n_layers)
    scores = [torch.from_numpy(rng.random((int(rng.integers(3, 60)), int(rng.integers(16, 70)))).astype(np.float32)).cuda()
              for _ in range(n_layers)]
    L, pp, i32 = tw.lib(), ctypes.POINTER(ctypes.c_void_p), ctypes.c_int32
    d = twprune._DeviceLayers(scores).make_masks()
    head = (n_layers, tw._ptr(d.K, i32), tw._ptr(d.N, i32), ctypes.cast(d.p_scores, pp))
    masks, thr, thr2 = ctypes.cast(d.p_masks, pp), ctypes.c_double(), (ctypes.c_double * 2)()
    never = tw.MASKS_READY(lambda d: 7)
    nothing = tw.MASKS_READY(lambda d: 0)
    calls = {  # entry point: its arguments, how they go on behind the masks, and how those of the _late form do
        "tiled_wise_1d": ((60.0, 0, 16), lambda ready: (masks, *ready, ctypes.byref(thr), d.stream)),
        "tiled_wise_2d": ((60.0, 0, 1, 16), lambda ready: (masks, *ready, None, thr2, d.stream)),
        "tiled_wise_1d_mix": ((65.0, 0, 16, 5.0, 0), lambda ready: (masks, *ready, ctypes.byref(thr), d.stream)),
    }
    for name, (args, rest) in calls.items():
        print("entry point", name, n_layers, flush=True)
        plain, late = getattr(L, "tw_prune_" + name), getattr(L, "tw_prune_" + name + "_late")
        want = getattr(twprune, name)(scores, 60, 16, return_device=True)
        for m in d.d_masks:
            m.fill_(9)
        assert plain(*head, *args, *rest(())) == 0
        assert all(torch.equal(a, b) for a, b in zip(want, d.d_masks))
        last = {"tiled_wise_1d": lambda: twprune.tiled_wise_1d.last_threshold, "tiled_wise_1d_mix": lambda: twprune.tw_mix_fn.last_threshold,
                "tiled_wise_2d": lambda: twprune.tiled_wise_2d.last_thresholds}[name]()
        assert last == (tuple(thr2) if name == "tiled_wise_2d" else thr.value)
        kept, d.p_masks[n_layers - 1] = d.p_masks[n_layers - 1], None
        assert plain(*head, *args, *rest(())) == tw.ERR_NULL
        assert late(*head, *args, *rest((nothing, None))) == tw.ERR_NULL
        d.p_masks[n_layers - 1] = kept
        assert late(*head, *args, *rest((never, None))) == tw.ERR_ALLOC
        for m in d.d_masks:
            m.fill_(9)
        assert plain(*head, *args, *rest(())) == 0
        assert all(torch.equal(a, b) for a, b in zip(want, d.d_masks))


def test_more_workgroups_than_a_launch_takes(tw, twprune):
    """2^24 workgroups of 256 threads, which one launch does not run: row norms of as many items, and thresholds of as
    many tiles."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(6)
    s = torch.rand((1 << 23, 64), generator=gen, device="cuda")  # 2^24 items of 32 rows of one column
    mask = twprune.tiled_wise_1d([s], 75, 1, return_device=True)[0].bool()
    assert s.masked_fill(~mask, 2.0).min() > s.masked_fill(mask, -1.0).max()
    assert abs(int(mask.sum()) - (1 << 27)) < 1000  # (equal values: some 32 of each)
    del s, mask
    tw.release_memory()
    s = np.random.default_rng(6).random((4, (1 << 24) + 3), dtype=np.float32)
    half = 1 << 23
    got = twprune.granularity_pruning(s, 40, 1)
    for part in (slice(0, half), slice(half, 2 * half), slice(2 * half, None)):
        assert np.array_equal(got[:, part], twprune.granularity_pruning(s[:, part], 40, 1))
    tw.release_memory()


@pytest.mark.parametrize("shapes", [[(20992, 4096)], [(10496, 8192), (33, 4)], [(20992, 4099)]])
def test_scores_beyond_the_caches(twprune, shapes):
    """More than 320 MB of scores are read past the caches, by either kernel of the row norms: the same masks
    as from the norms and the percentile one at a time."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(5)
    scores = [torch.randn(s, generator=gen, device="cuda").abs_() for s in shapes]
    got = twprune.tiled_wise_1d(scores, 75, 128, return_device=True)
    norms = [twprune.tile_row_norms(s.cpu().numpy(), twprune.tiles_every_g_columns(s.shape[1], 128)) for s in scores]
    thr = twprune.percentile(np.concatenate([n.ravel() for n in norms]), 75)
    for s, n, m in zip(scores, norms, got):
        keep = torch.from_numpy(n > thr).cuda().t().repeat_interleave(128, 1)[:, :s.shape[1]]
        assert torch.equal(m.bool(), keep)
