"""GPU parity of the mixed (TW + element-wise remainder) producers, tw_prune_mix through the C
ABI, against the golden vectors of the reference's prune_algo.py:151-193 and the CPU oracle;
and of the covering plan that runs such masks on the TW kernel.

Masks: bit-exact.  GEMM on a covering plan: max relative error <= 1e-2 (fp16) / 2e-2 (bf16)
against the float64 product of the 16-bit operands with the mask applied."""
import json
import os

import numpy as np
import pytest

from tests.test_gpu_gemm import run_gemm

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


def parse(text):
    return int(text) if text.lstrip("-").isdigit() else float(text)


def test_golden_vectors_mix(twprune):
    z = np.load(GOLD)
    meta = json.loads(bytes(z["meta"]).decode())
    for case in meta["cases"]:
        name, g = case["name"], case["granularity"]
        scores = twprune.img2col_forward([z["%s/w%d" % (name, i)] for i in range(len(case["shapes"]))])
        for fn, sp, g1 in meta["mix"][name]:
            print("case", name, fn, sp, g1, flush=True)
            got = getattr(twprune, fn)(scores, parse(sp), g, parse(g1))
            for i, m in enumerate(got):
                want = np.unpackbits(z["%s/%s/%s/%s/m%d" % (name, fn, sp, g1, i)])[:m.size]
                assert np.array_equal(m.ravel(), want.astype(bool)), (name, fn, sp, g1, i)


SHAPES = [
    [(64, 256), (128, 384)],
    [(100, 130), (33, 500), (257, 64)],
    [(3, 3, 16, 48), (48, 72)],
    [(1, 1)],
]


@pytest.mark.parametrize("shapes", SHAPES)
@pytest.mark.parametrize("g1", [5, 1, 2.5, 0, np.float64(3.0)])
def test_mix_matches_oracle(twprune, po, shapes, g1):
    rng = np.random.default_rng(abs(hash((str(shapes), float(g1)))) % 2 ** 31)
    scores = twprune.img2col_forward([rng.standard_normal(s).astype(np.float32) for s in shapes])
    for sp, g in ((75, 32), (50.0, 128), (90, 8)):
        print("mix", shapes, repr(g1), sp, g, flush=True)
        for fn in ("tiled_wise_1d_mix", "tiled_wise_2d_mix"):
            want = getattr(po, fn)(scores, sp, g, g1)
            got = getattr(twprune, fn)(scores, sp, g, g1)
            for w, m in zip(want, got):
                assert np.array_equal(w, m), (fn, sp, g)
    # the second stage alone, on masks that are not tile-wise at all
    masks = [rng.random(s.shape) < 0.3 for s in scores]
    want, thr = po.tw_mix_fn(scores, g1, masks)
    got = twprune.tw_mix_fn(scores, g1, masks)
    assert np.float64(thr) == twprune.tw_mix_fn.last_threshold
    for w, m in zip(want, got):
        assert np.array_equal(w, m)


def test_mix_ties_and_extremes(twprune, po):
    rng = np.random.default_rng(41)
    scores = [(np.round(rng.standard_normal((96, 128)) * 2) / 2).astype(np.float32) for _ in range(2)]
    scores = twprune.img2col_forward(scores)
    for sp, g1 in ((50, 5), (0, 100), (95, 5), (60, 33.3), (99, 1)):
        want = po.tiled_wise_1d_mix(scores, sp, 16, g1)
        got = twprune.tiled_wise_1d_mix(scores, sp, 16, g1)
        for a, b in zip(want, got):
            assert np.array_equal(a, b), (sp, g1)


@pytest.mark.parametrize("values", ["normal", "few_values", "mostly_zero", "extreme_scales"])
def test_mix_selection_narrowed_by_a_sample(twprune, po, values):
    """Enough elements for the sampled bracket (more than 2^17): it holds the threshold ("normal"), or
    it cannot be narrow because the values around the threshold repeat ("few_values",
    "mostly_zero") and the selection walks all elements; squares that leave the normal range
    ("extreme_scales") take the square root.  Masks are integers: bit for bit the oracle's."""
    rng = np.random.default_rng(43)
    shapes = [(577, 300), (64, 1000), (33, 7)]     # whole items, ragged ones, a layer off 16 bytes
    w = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    if values == "few_values":
        w = [(np.round(x * 2) / 2).astype(np.float32) for x in w]
    elif values == "mostly_zero":
        w = [np.where(rng.random(x.shape) < 0.9, 0, x).astype(np.float32) for x in w]
    elif values == "extreme_scales":
        w = [(x * 10.0 ** rng.integers(-25, 18, x.shape)).astype(np.float32) for x in w]
    scores = twprune.img2col_forward(w)
    masks = [rng.random(s) < 0.3 for s in shapes]
    for g1 in (5, 0.01, 50, 100):
        want, thr = po.tw_mix_fn(scores, g1, masks)
        got = twprune.tw_mix_fn(scores, g1, masks)
        assert np.float64(thr) == twprune.tw_mix_fn.last_threshold, (values, g1)
        for a, b in zip(want, got):
            assert np.array_equal(a, b), (values, g1)


@pytest.mark.parametrize("g1", [50, 9.76, 7])       # the rank among normal scores, below an infinite one, among those
def test_mix_nan_beside_huge_values(twprune, g1):
    """A NaN next to a score whose square overflows: every element's score is its own, sqrt(x x), whatever
    stands beside it.  NaNs rank above everything; the expectation is NumPy's float32 arithmetic on that order."""
    rng = np.random.default_rng(44)
    x = rng.random((64, 64)).astype(np.float32)
    flat = x.reshape(-1)
    flat[0:800:4], flat[1:800:4] = 1e20, np.nan        # 200 neighbouring pairs, each in one lane's group
    mask0 = np.zeros(x.shape, bool)
    with np.errstate(over="ignore", invalid="ignore"):
        score = np.sqrt(flat * flat)
        s = np.sort(score)                             # (NaNs last)
        virt = np.float32(s.size - 1) * (np.float32(100 - g1) / np.float32(100))
        k = int(np.floor(virt))
        g, a, b = np.float32(virt - np.floor(virt)), s[k], s[k + 1]
        thr = b - (b - a) * (np.float32(1) - g) if g >= 0.5 else a + (b - a) * g
        want = (score > thr).reshape(x.shape)
    got = twprune.tw_mix_fn([x], g1, [mask0])[0]
    assert np.array_equal(np.float64(thr), np.float64(twprune.tw_mix_fn.last_threshold), equal_nan=True)
    assert np.array_equal(want, got)


def test_mix_error_paths(tw, twprune):
    with pytest.raises(tw.TwError):
        twprune.tiled_wise_1d_mix([np.ones((4, 4), np.float32)], 50, 2, 120)   # percentile < 0
    with pytest.raises(tw.TwError):
        twprune.tiled_wise_1d_mix([np.ones((4, 4), np.float32)], 98, 2, 5)     # TW stage > 100


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_cover_plan_runs_mixed_masks(tw, twprune, po, oracle, dtype):
    """A mixed mask is not tile-wise (the plain builder refuses it); the covering plan computes
    A (B (.) mask) exactly as masked, and its lists are the union of each tile's elements."""
    rng = np.random.default_rng(42)
    K, N, G, M = 320, 384, 128, 200
    W = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    # structured magnitudes, so that the remainder does not touch every row of every tile
    W *= (rng.random((K, 1)) < 0.5) * 0.9 + 0.1
    scores = twprune.img2col_forward([W])
    mask = twprune.tiled_wise_1d_mix(scores, 70, G, 2)[0]
    table = po.tiles_every_g_columns(N, G)
    with pytest.raises(tw.TwError) as e:
        tw.Plan.from_mask_tiles(mask, table, dtype, W)
    assert e.value.status == tw.ERR_NOT_TW
    with tw.Plan.from_mask_tiles(mask, table, dtype, W, cover=True) as plan:
        ex, _ = plan.export(with_weight=False)
        want = po.cover_tiles_from_mask(mask, table)
        for t, wt in zip(ex, want):
            assert t["kept_k"].tolist() == wt["kept_k"] and t["kept_n"].tolist() == wt["kept_n"]
        A = rng.standard_normal((M, K)).astype(np.float32)
        C, _ = run_gemm(tw, oracle, plan, A, dtype, N, pruned=1)
        ref = oracle.quantize(A, dtype).astype(np.float64) @ (oracle.quantize(W, dtype) * mask).astype(np.float64)
        assert oracle.rel_error(C, ref) <= (1e-2 if dtype == "f16" else 2e-2)
    # a tile-wise mask gives the same plan with and without `cover`
    m1 = twprune.tiled_wise_1d(scores, 70, G)[0]
    with tw.Plan.from_mask_tiles(m1, table, dtype, W) as p1, \
            tw.Plan.from_mask_tiles(m1, table, dtype, W, cover=True) as p2:
        (t1, b1), (t2, b2) = p1.export(), p2.export()
        assert np.array_equal(b1, b2)
        for a, b in zip(t1, t2):
            assert np.array_equal(a["kept_k"], b["kept_k"]) and np.array_equal(a["kept_n"], b["kept_n"])


VGG16_LAYERS = [(27, 64), (576, 64), (576, 128), (1152, 128), (1152, 256), (2304, 256), (2304, 256),
                (2304, 512), (4608, 512), (4608, 512), (4608, 512), (4608, 512), (4608, 512),
                (4096, 4096)]


def test_full_size_network_all_producers(twprune, po):
    """A VGG16-sized list of score matrices (31.6 M elements, the 13 conv layers as im2col
    matrices and one 4096 x 4096 dense layer): every producer returns the oracle's masks bit for
    bit, and the kept fractions are the requested ones."""
    rng = np.random.default_rng(20200615)
    scores = [np.abs(rng.standard_normal(s)).astype(np.float32) for s in VGG16_LAYERS]
    total = sum(k * n for k, n in VGG16_LAYERS)
    print("full size: 1d", flush=True)
    want, _, _ = po.tiled_wise_1d(scores, 75, 128)
    got = twprune.tiled_wise_1d(scores, 75, 128)
    assert all(np.array_equal(w, g) for w, g in zip(want, got))
    assert abs(sum(int(g.sum()) for g in got) / total - 0.25) < 0.01
    print("full size: 2d", flush=True)
    want = po.tiled_wise_2d(scores, 75, 128)[0]
    got = twprune.tiled_wise_2d(scores, 75, 128)
    assert all(np.array_equal(w, g) for w, g in zip(want, got))
    print("full size: 1d mix", flush=True)
    want = po.tiled_wise_1d_mix(scores, 75, 128, 5)
    got = twprune.tiled_wise_1d_mix(scores, 75, 128, 5)
    assert all(np.array_equal(w, g) for w, g in zip(want, got))
    # TW at 80 % plus the top 5 % of the shifted element scores: between 20 % and 25 % kept
    kept = sum(int(g.sum()) for g in got) / total
    assert 0.20 < kept <= 0.2501
    print("full size: 2d mix", flush=True)
    want = po.tiled_wise_2d_mix(scores, 75, 128, 1)
    got = twprune.tiled_wise_2d_mix(scores, 75, 128, 1)
    assert all(np.array_equal(w, g) for w, g in zip(want, got))



@pytest.mark.parametrize("g1", [5, 50])
def test_mix_selection_with_uneven_pieces(twprune, po, g1):
    """The values inside the bracket lie together: a third of a few thousand consecutive elements, so that the pieces of the waves
    that read these hold some three hundred values each and most others few or none.  Bit for bit the oracle's."""
    rng = np.random.default_rng(47)
    shapes = [(577, 300), (64, 1000), (33, 7)]
    scores = [np.abs(rng.standard_normal(s)).astype(np.float32) for s in shapes]
    masks = [np.zeros(s, bool) for s in shapes]
    flat = scores[0].reshape(-1)
    at = np.quantile(np.concatenate([s.reshape(-1) for s in scores]), 1 - g1 / 100)
    near = np.flatnonzero(rng.random(20480) < 0.35) + 8192
    flat[near] = at * (1 + 0.002 * (rng.random(near.size) - 0.5))
    want, thr = po.tw_mix_fn(scores, g1, masks)
    got = twprune.tw_mix_fn(scores, g1, masks)
    assert np.float64(thr) == twprune.tw_mix_fn.last_threshold
    for a, b in zip(want, got):
        assert np.array_equal(a, b)

def _mixed_layer(rng, twprune, K, N, G, sparsity, g1, structured):
    """Weight, the TW mask of the mixed producer's first stage and the mixed mask."""
    W = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    if structured:
        W *= (rng.random((K, 1)) < 0.5) * 0.9 + 0.1
    scores = twprune.img2col_forward([W])
    mask = twprune.tiled_wise_1d_mix(scores, sparsity, G, g1)[0]
    mask0 = twprune.tiled_wise_1d(scores, sparsity + g1, G)[0]
    assert not (mask0 & ~mask).any()          # the mixed mask only adds elements
    return W, mask0, mask


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M", [200, 513, 2100, 4300])
def test_side_kernel_runs_the_remainder(tw, twprune, po, oracle, dtype, M):
    """TW plan of the first stage's mask + tw_side_gemm on what the second stage adds = the masked
    layer A (B (.) mask) of the mixed mask.  The two passes round their results to 16 bits one
    after the other, so an element's error is relative to the larger of the tile-wise part and
    the sum (where the remainder cancels the tile-wise part, the first rounding stays): within
    the GEMM tolerance of the float64 products of the 16-bit operands on that scale.  The side
    call alone adds exactly the remainder's product (checked against a launch on zeros, one
    rounding: plain relative error), leaves columns without remainder elements and the padding
    beyond M untouched, and repeats bit for bit.  A die takes whole 256-row chunks in rounds of
    eight and the chunks left over are shared: M = 200 and 513 have left-over chunks only, 2100
    (nine chunks) one round and one left over, 4300 (seventeen) two rounds and one left over."""
    import torch
    from tests.test_gpu_gemm import to_device_bits, from_device_bits, round_up, SENTINEL
    rng = np.random.default_rng(77 + M)
    K, N, G = 320, 384, 128
    W, mask0, mask = _mixed_layer(rng, twprune, K, N, G, 70, 2, structured=True)
    rem = mask & ~mask0
    rem[:, 5] = False                          # a column without remainder elements
    rem[:, 300:310] = False
    mask = mask0 | rem
    table = po.tiles_every_g_columns(N, G)
    A = rng.standard_normal((M, K)).astype(np.float32)
    lda = ldc = round_up(M, 8) + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)
    s = torch.cuda.current_stream().cuda_stream
    tol = 1e-2 if dtype == "f16" else 2e-2
    with tw.Plan.from_mask_tiles(mask0, table, dtype, W) as plan, tw.Side(rem, dtype, W) as side:
        assert side.nnz == int(rem.sum())
        outs = []
        for rep in range(2):
            dC = to_device_bits(np.full((N, ldc), SENTINEL, np.uint16), (N, ldc))
            print("side test: plan + side", M, dtype, rep, flush=True)
            plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, pruned_cols=tw.PRUNED_ZERO, stream=s)
            side.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, stream=s)
            torch.cuda.synchronize()
            outs.append(from_device_bits(dC))
        assert np.array_equal(outs[0], outs[1])
        assert (outs[0][:, M:] == SENTINEL).all()
        C = oracle.bits_to_f32(outs[0][:, :M], dtype).reshape(N, M).T
        Aq, Wq = oracle.quantize(A, dtype).astype(np.float64), oracle.quantize(W, dtype).astype(np.float64)
        ref, ref_tw = Aq @ (Wq * mask), Aq @ (Wq * mask0)
        floor = 1e-2 * np.sqrt(np.mean(ref * ref))
        assert np.max(np.abs(C - ref) / np.maximum(np.maximum(np.abs(ref), np.abs(ref_tw)), floor)) <= tol
        # the side call alone, on zeros, with alpha: exactly alpha * A (W (.) rem), one rounding
        dZ = to_device_bits(np.zeros((N, ldc), np.uint16), (N, ldc))
        side.gemm(dA.data_ptr(), dZ.data_ptr(), M, lda=lda, ldc=ldc, alpha=-0.5, stream=s)
        torch.cuda.synchronize()
        Z = from_device_bits(dZ)
        untouched = ~rem.any(axis=0)
        assert (Z[untouched] == 0).all() and (Z[:, M:] == 0).all()
        Zf = oracle.bits_to_f32(Z[:, :M], dtype).reshape(N, M).T
        assert oracle.rel_error(Zf, -0.5 * (Aq @ (Wq * rem))) <= tol


def test_side_edge_cases_and_errors(tw):
    import torch
    K, N, M = 64, 40, 16
    W = np.ones((K, N), np.float32)
    dA = torch.ones((K, M), dtype=torch.float16, device="cuda")
    dC = torch.full((N, M), 3.0, dtype=torch.float16, device="cuda")
    with tw.Side(np.zeros((K, N), bool), "f16", W) as side:       # an empty remainder does nothing
        assert side.nnz == 0
        side.gemm(dA.data_ptr(), dC.data_ptr(), M)
        torch.cuda.synchronize()
        assert (dC == 3.0).all()
    full = np.ones((K, N), bool)
    with tw.Side(full, "f16", W) as side:                         # every element: a dense product
        assert side.nnz == K * N
        side.gemm(dA.data_ptr(), dC.data_ptr(), 0)                # M = 0: nothing
        side.gemm(dA.data_ptr(), dC.data_ptr(), M)
        torch.cuda.synchronize()
        assert (dC == 3.0 + K).all()
        with pytest.raises(tw.TwError):
            side.gemm(0, dC.data_ptr(), M)
        with pytest.raises(tw.TwError):
            side.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=M - 8)
        with pytest.raises(tw.TwError):
            side.gemm(dA.data_ptr(), dC.data_ptr(), M, ldc=M + 4)
        with pytest.raises(tw.TwError):
            side.gemm(dA.data_ptr() + 2, dC.data_ptr(), M)
    with pytest.raises(ValueError):
        tw.Side(full, "f16", W[:, :3])


@pytest.mark.parametrize("values", ["normal", "few_values", "huge"])
@pytest.mark.parametrize("granularity", [128, 5, 2, 1000])
def test_1d_mix_in_one_call(twprune, po, granularity, values):
    """The masks without those of the first stage between the two: rows of whole and of odd numbers of fours,
    tiles whose last one is one or two columns wide (no vectors), a layer off 16 bytes, layers of less than an
    item and of whole items; the bracket holds the threshold, or misses (repeated values, the largest or next to
    nothing kept beside the tiles) and the masks are made again from what the narrowing pass left."""
    import torch
    rng = np.random.default_rng(46)
    shapes = [(512, 384), (577, 301), (64, 1002), (4096, 3), (9, 7)]
    w = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    if values == "few_values":
        w = [(np.round(x * 2) / 2).astype(np.float32) for x in w]
    elif values == "huge":  # one square in fifty overflows: infinite scores, and a threshold among them
        w = [np.where(rng.random(x.shape) < 0.02, x * 1e25, x).astype(np.float32) for x in w]
    scores = twprune.img2col_forward(w)
    dev = [torch.from_numpy(x).cuda() for x in scores]
    off = torch.empty(dev[1].numel() + 1, device="cuda")[1:].view(dev[1].shape)  # starts 4 bytes behind a piece of 16
    off.copy_(dev[1])
    dev[1] = off
    for sp, g1 in ((75, 5), (60.0, np.float64(12.5)), (90, 0.01), (40, 60), (50, 0)):
        with np.errstate(all="ignore"):
            want = po.tiled_wise_1d_mix(scores, sp, granularity, g1)
        got = twprune.tiled_wise_1d_mix(dev, sp, granularity, g1, return_device=True)
        for a, b in zip(want, got):
            assert np.array_equal(np.asarray(a, bool), b.cpu().numpy().astype(bool)), (sp, g1, a.shape)
            assert b.max() <= 1


@pytest.mark.parametrize("granularity", [4, 100, 128])
@pytest.mark.parametrize("values", ["normal", "tiny", "huge", "no_numbers"])
def test_mix_bracket_of_whole_fours(twprune, granularity, values):
    """Four neighbours in one row of one tile (no layer asks for the kernel that looks at two), items in vectors and
    without, and scores that the bracket is compared with as bits: below and above the range where sqrt(x x) is |x| again,
    infinite ones and NaNs, which rank above everything and are in no mask.  The expectation is NumPy's float32 arithmetic on the
    masks of the first stage."""
    import torch
    rng = np.random.default_rng(47)
    scores = [np.abs(rng.standard_normal(s)).astype(np.float32) for s in ((512, 384), (577, 300), (64, 1000), (9, 8))]
    with np.errstate(all="ignore"):
        if values == "tiny":
            scores = [(x * 10.0 ** rng.integers(-26, -16, x.shape)).astype(np.float32) for x in scores]
        elif values == "huge":
            scores = [(x * 10.0 ** rng.integers(16, 22, x.shape)).astype(np.float32) for x in scores]
        elif values == "no_numbers":
            for x in scores[:3]:
                at = rng.permutation(x.size)[:60]
                x.reshape(-1)[at[:30]], x.reshape(-1)[at[30:]] = np.inf, np.nan
    dev = [torch.from_numpy(x).cuda() for x in scores]
    for sp, g1 in ((75, 5), (60, 1), (50, 40)):
        first = twprune.tiled_wise_1d(dev, sp + g1 if sp + g1 <= 100 else 100, granularity, return_device=True)
        masks = [m.cpu().numpy() != 0 for m in first]
        with np.errstate(all="ignore"):
            own = [np.sqrt(x * x) - m.astype(np.float32) for x, m in zip(scores, masks)]
            s = np.sort(np.concatenate([v.reshape(-1) for v in own]))  # (NaNs last)
            virt = np.float32(s.size - 1) * (np.float32(100 - g1) / np.float32(100))
            k = int(np.floor(virt))
            g, a, b = np.float32(virt - np.floor(virt)), s[k], s[k + 1]
            thr = b - (b - a) * (np.float32(1) - g) if g >= 0.5 else a + (b - a) * g
            want = [m | (v > thr) for m, v in zip(masks, own)]
        for got in (twprune.tiled_wise_1d_mix(dev, sp, granularity, g1, return_device=True),
                    twprune.tw_mix_fn(dev, g1, first, return_device=True)):
            assert np.array_equal(np.float64(thr), np.float64(twprune.tw_mix_fn.last_threshold), equal_nan=True), (sp, g1)
            for x, y in zip(want, got):
                assert np.array_equal(x.astype(np.uint8), y.cpu().numpy()), (sp, g1, x.shape)


@pytest.mark.parametrize("K,N,granularity", [(5, 1 << 21, 128), (5, 1 << 21, 3), (4, (1 << 21) - 1, 3), (4, (1 << 21) - 2, 3),
                                             (3, (1 << 21) + 8, 128), (1 << 23, 4, 4), (1 << 23, 3, 2), ((1 << 23) + 1, 4, 4),
                                             (1 << 23, 64, 1)])
def test_1d_mix_at_its_limits(tw, twprune, K, N, granularity):
    """The widest and the tallest layer whose elements are placed in rows and tiles by a multiplication in float and by
    24-bit products, the most norms, and the first layers beyond, where one stage follows the other with the masks as
    input and output: the masks of the two calls, whose kernels divide."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(K + N)
    scores = [torch.rand((K, N), generator=gen, device="cuda"), torch.rand((64, 100), generator=gen, device="cuda")]
    for sp, g1 in ((75, 5), (40, 0.5)):
        want = twprune.tw_mix_fn(scores, g1, twprune.tiled_wise_1d(scores, sp + g1, granularity, return_device=True), return_device=True)
        threshold = twprune.tw_mix_fn.last_threshold
        got = twprune.tiled_wise_1d_mix(scores, sp, granularity, g1, return_device=True)
        assert twprune.tw_mix_fn.last_threshold == threshold
        assert all(torch.equal(a, b) for a, b in zip(want, got)), (sp, g1)
        del want, got
    tw.release_memory()
