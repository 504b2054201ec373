"""The weight-stationary kernel (TW_SHAPE_BS: a unit's packed weight in registers, the kept rows of A
streamed through LDS by loads that write LDS directly) against the streaming 256 x 128 kernel, bit
for bit, and against the oracle (max relative error 1e-2 fp16 / 2e-2 bf16).  It takes plans whose
tiles keep at most 192 rows, K-major operands and beta == 0; a forced shape it does not take falls
back to the automatic choice."""
import numpy as np
import pytest

from tests.helpers import from_device_bits, to_device_bits

pytestmark = pytest.mark.gpu

TOL = {"f16": 1e-2, "bf16": 2e-2}
SENTINEL = 0x1234


def make_tiles(rng, K, G, spec):
    tiles = []
    for t, (kt, nt) in enumerate(spec):
        tiles.append(dict(col0=t * G, width=G,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(G, size=nt, replace=False)).astype(np.int32)))
    return tiles


CASES = [
    # M, K, G, (kept rows, kept columns) per tile
    (333, 700, 128, ((192, 128), (64, 100), (0, 128), (191, 128), (130, 7), (1, 33))),    # up to three steps
    (1000, 300, 128, ((128, 128), (65, 96), (100, 128))),                                  # two steps
    (4100, 520, 64, ((190, 64), (3, 51), (129, 33), (0, 10), (64, 64))),                   # three steps, G = 64
    (64, 200, 32, ((10, 32), (70, 20))),                                                   # one range, few rows
    (2500, 256, 128, tuple((60 + 3 * t, 128 - t) for t in range(40))),                     # more units than argument slots
]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_weight_stationary_kernel(tw, oracle, dtype, case):
    import torch
    M, K, G, spec = CASES[case]
    N = G * len(spec)
    rng = np.random.default_rng(900 + case)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = make_tiles(rng, K, G, spec)
    keep = np.zeros(N, bool)
    for t in tiles:
        keep[t["col0"] + t["kept_n"]] = True
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = (M + 7) // 8 * 8 + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)
    s = torch.cuda.current_stream().cuda_stream

    def launch(plan, shape, alpha, pruned, with_bias, act, per_cu=-1):
        dC = torch.full((N, ldc), SENTINEL, dtype=torch.int16, device="cuda")
        tw.set_option(tw.OPT_SHAPE, shape)
        tw.set_option(tw.OPT_WGS_PER_CU, per_cu)
        print("weight-stationary test: case", case, "shape", shape, alpha, pruned, with_bias, act, per_cu, dtype, flush=True)
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, pruned_cols=pruned,
                  bias_ptr=dbias.data_ptr() if with_bias else None, activation=act, stream=s)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, pruned, with_bias, act) in ((1.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                                                    (0.5, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                                                    (1.0, tw.PRUNED_ZERO, True, tw.ACT_TANH)):
                want = launch(plan, tw.SHAPE_256x128, alpha, pruned, with_bias, act)
                for per_cu in (-1, 1, 8):     # few and many ranges of rows
                    got = launch(plan, tw.SHAPE_BS, alpha, pruned, with_bias, act, per_cu)
                    if act == tw.ACT_TANH:
                        a = oracle.bits_to_f32(got[:, :M], dtype)
                        b = oracle.bits_to_f32(want[:, :M], dtype)
                        assert oracle.rel_error(a, b) <= 0.5 * TOL[dtype]
                        assert np.array_equal(got[:, M:], want[:, M:])
                    else:
                        assert np.array_equal(got, want), (alpha, pruned, with_bias, act, per_cu)
                    again = launch(plan, tw.SHAPE_BS, alpha, pruned, with_bias, act, per_cu)
                    assert np.array_equal(got, again)
                if not with_bias:
                    Cf = oracle.bits_to_f32(got[:, :M], dtype).reshape(N, M).T
                    ref = oracle.stream_gemm_nn(oracle.quantize(A, dtype), oracle.quantize(B, dtype), tiles, alpha)
                    assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
                    assert np.all(got[~keep, :] == SENTINEL) and np.all(got[:, M:] == SENTINEL)
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
        tw.set_option(tw.OPT_WGS_PER_CU, -1)


def test_weight_stationary_kernel_declines(tw, oracle):
    """Tiles with more than 192 kept rows, or beta != 0: the forced shape does not apply and the
    launch runs what it would have run anyway (same bits as the automatic choice)."""
    import torch
    rng = np.random.default_rng(77)
    M, K, G = 300, 600, 128
    tiles = make_tiles(rng, K, G, ((300, 128), (100, 128)))
    N = 2 * G
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    At = np.ascontiguousarray(oracle.cast_bits(A, "f16").reshape(M, K).T)
    ld = 304
    Ap = np.zeros((K, ld), np.uint16)
    Ap[:, :M] = At
    dA = to_device_bits(Ap, Ap.shape)
    s = torch.cuda.current_stream().cuda_stream
    out = []
    try:
        with tw.Plan.create(K, N, "f16", tiles, B) as plan:
            for shape in (-1, tw.SHAPE_BS):
                tw.set_option(tw.OPT_SHAPE, shape)
                dC = torch.zeros((N, ld), dtype=torch.int16, device="cuda")
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=ld, ldc=ld, stream=s)
                torch.cuda.synchronize()
                out.append(from_device_bits(dC).copy())
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
    assert np.array_equal(out[0], out[1])


# M, K, G, (kept rows, kept columns) per tile: the wider form where the launch takes it by itself, one to six steps, units of one
# to four blocks of columns, tiles without a kept row, ranges of two blocks of 64 rows and of many, M off every grain; the last
# one's output is stored in lines
WIDE_CASES = [
    (4101, 1100, 128, ((256, 128), (200, 100), (0, 128), (255, 65), (193, 7), (220, 33))),
    (1031, 1200, 128, ((384, 128), (257, 97), (321, 32), (0, 5), (380, 128)) * 5),
    (97, 600, 128, tuple((300 + t % 64, 128 if t % 3 else 64) for t in range(256))),
    (2600, 1100, 128, tuple((230 + 13 * (t % 12), 128 - t) for t in range(40))),
    (6001, 130, 128, tuple((60 + t % 68, 128 - t % 31) for t in range(64))),
]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("case", range(len(WIDE_CASES)))
def test_weight_stationary_wide_form(tw, oracle, dtype, case):
    """Bit for bit the streaming 256 x 128 kernel (both add a tile's kept rows up in the order of its list, in fp32), with every
    activation and either treatment of the pruned columns, the padding of C's rows untouched.  GELU and tanh: the kernels build
    them from the same sum in a different order of instructions, so one unit in the last place of the result (2^-10, 2^-7)."""
    import torch
    M, K, G, spec = WIDE_CASES[case]
    N = G * len(spec)
    rng = np.random.default_rng(1300 + case)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    dbias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).cuda()
    tiles = make_tiles(rng, K, G, spec)
    used = np.unique(np.concatenate([t["kept_k"] for t in tiles]))
    lda = ldc = (M + 7) // 8 * 8 + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    At[np.setdiff1d(np.arange(K), used)] = 0x7fff       # NaN in the rows that no tile keeps: they reach no product
    dA = to_device_bits(At, At.shape)
    s = torch.cuda.current_stream().cuda_stream
    tdt = torch.float16 if dtype == "f16" else torch.bfloat16
    ulp = 2.0 ** -10 if dtype == "f16" else 2.0 ** -7

    def launch(plan, shape, alpha, pruned, with_bias, act):
        dC = torch.full((N, ldc), SENTINEL, dtype=torch.int16, device="cuda")
        tw.set_option(tw.OPT_SHAPE, shape)
        print("wide form: case", case, "shape", shape, alpha, pruned, with_bias, act, dtype, flush=True)
        assert plan.choice(M, lda=lda, ldc=ldc)["shape"] == (tw.SHAPE_BS if shape == -1 else shape)
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, pruned_cols=pruned,
                  bias_ptr=dbias.data_ptr() if with_bias else None, activation=act, stream=s)
        torch.cuda.synchronize()
        return dC

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, pruned, with_bias, act) in ((1.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                                                    (0.5, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                                                    (1.0, tw.PRUNED_ZERO, True, tw.ACT_GELU),
                                                    (1.0, tw.PRUNED_UNTOUCHED, True, tw.ACT_TANH)):
                want = launch(plan, tw.SHAPE_256x128, alpha, pruned, with_bias, act)
                got = launch(plan, -1, alpha, pruned, with_bias, act)
                if act in (tw.ACT_GELU, tw.ACT_TANH):
                    a, b = got[:, :M].view(tdt).float(), want[:, :M].view(tdt).float()
                    assert bool(((a - b).abs() <= ulp * b.abs() + 1e-7).all())
                    assert torch.equal(got[:, M:], want[:, M:])
                else:
                    assert torch.equal(got, want), (alpha, pruned, with_bias, act)
                assert torch.equal(got, launch(plan, -1, alpha, pruned, with_bias, act))
            if case == 2:   # (the smallest)
                out = from_device_bits(launch(plan, -1, 1.0, tw.PRUNED_ZERO, False, tw.ACT_NONE))
                keep = np.zeros(N, bool)
                for t in tiles:
                    keep[t["col0"] + t["kept_n"]] = True
                ref = oracle.stream_gemm_nn(oracle.quantize(A, dtype), oracle.quantize(B, dtype), tiles, 1.0)
                Cf = oracle.bits_to_f32(out[:, :M], dtype).reshape(N, M).T
                assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
                assert not Cf[:, ~keep].any()
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


@pytest.mark.parametrize("kept", [100, 350])
def test_weight_stationary_padding_lies_beyond_the_largest_a(tw, oracle, kept):
    """The padding of a tile's row list is fetched from beyond A's buffer, which delivers zeros - also where A ends 16 bytes
    short of 4 GiB: NaN in the last 256 bytes of A (padding behind row K - 1) reaches no product.  Bit for bit what the same
    rows of A give in a small buffer."""
    import torch
    M, K, G, N = 4096, 3741, 128, 1024
    rng = np.random.default_rng(91 + kept)
    tiles = make_tiles(rng, K - 1, G, ((kept, G),) * (N // G))
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    Ab = torch.randn((K, M), generator=torch.Generator("cuda").manual_seed(kept), device="cuda").half()
    s = torch.cuda.current_stream().cuda_stream
    out = []
    with tw.Plan.create(K, N, "f16", tiles, B) as plan:
        for lda in (M, 574040):
            dA = torch.zeros((K, lda), dtype=torch.float16, device="cuda")
            dA[:, :M] = Ab
            if lda > M:
                assert dA.numel() * 2 == 2 ** 32 - 16
                dA[K - 1, lda - 128:] = float("nan")
            assert plan.choice(M, lda=lda, ldc=M)["shape"] == tw.SHAPE_BS
            dC = torch.zeros((N, M), dtype=torch.float16, device="cuda")
            print("padding beyond A: kept", kept, "lda", lda, flush=True)
            plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=M, stream=s)
            torch.cuda.synchronize()
            out.append(dC.view(torch.int16))
            del dA
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("case", range(len(CASES) + len(WIDE_CASES)))
def test_both_weight_stationary_kernels(tw, oracle, dtype, case):
    """The kernel of four multiplying waves (up to 192 kept rows) and the one of eight (up to 384), forced in turn: without
    activation and with ReLU bit for bit the streaming 256 x 128 kernel, with GELU and tanh one unit in the last place of the
    result (2^-10, 2^-7: the same sum, its activation from a different order of instructions), pruned columns filled and
    left alone, few and many ranges of rows, C's columns at sectors of memory and off them, the padding of its rows untouched."""
    import torch
    M, K, G, spec = (CASES + WIDE_CASES)[case]
    N = G * len(spec)
    rng = np.random.default_rng(1700 + case)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    dbias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).cuda()
    tiles = make_tiles(rng, K, G, spec)
    lda = (M + 7) // 8 * 8 + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)
    s = torch.cuda.current_stream().cuda_stream
    tdt = torch.float16 if dtype == "f16" else torch.bfloat16
    ulp = 2.0 ** -10 if dtype == "f16" else 2.0 ** -7
    names = {tw.SHAPE_BS4: "tw_gemm_bs_kernel", tw.SHAPE_BS8: "tw_gemm_bw_kernel", tw.SHAPE_256x128: "tw_gemm_ws_kernel 256x128"}

    def launch(plan, shape, ldc, pruned, act, per_cu=-1):
        dC = torch.full((N, ldc), SENTINEL, dtype=torch.int16, device="cuda")
        tw.set_option(tw.OPT_SHAPE, shape)
        tw.set_option(tw.OPT_WGS_PER_CU, per_cu)
        print("weight-stationary kernels: case", case, "shape", shape, ldc, pruned, act, per_cu, dtype, flush=True)
        assert plan.kernel_name(M, lda, ldc, activation=act) == names[shape]
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=0.5, pruned_cols=pruned, bias_ptr=dbias.data_ptr(),
                  activation=act, stream=s)
        torch.cuda.synchronize()
        return dC

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            sectors, off = (M + 31) // 32 * 32, (M + 7) // 16 * 16 + 8
            for ldc, pruned, act in ((off, tw.PRUNED_UNTOUCHED, tw.ACT_NONE), (sectors, tw.PRUNED_ZERO, tw.ACT_RELU),
                                     (sectors, tw.PRUNED_UNTOUCHED, tw.ACT_NONE), (off, tw.PRUNED_ZERO, tw.ACT_GELU),
                                     (sectors, tw.PRUNED_UNTOUCHED, tw.ACT_TANH)):
                want = launch(plan, tw.SHAPE_256x128, ldc, pruned, act)
                for shape in (tw.SHAPE_BS4, tw.SHAPE_BS8):
                    if shape == tw.SHAPE_BS4 and max(kt for kt, _ in spec) > 192:
                        continue
                    for per_cu in (-1, 1, 4):
                        got = launch(plan, shape, ldc, pruned, act, per_cu)
                        if act in (tw.ACT_GELU, tw.ACT_TANH):
                            a, b = got[:, :M].view(tdt).float(), want[:, :M].view(tdt).float()
                            assert bool(((a - b).abs() <= ulp * b.abs() + 1e-7).all())
                            assert torch.equal(got[:, M:], want[:, M:])
                        else:
                            assert torch.equal(got, want), (shape, pruned, act, per_cu)
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
        tw.set_option(tw.OPT_WGS_PER_CU, -1)


@pytest.mark.parametrize("M,N,kept,act,kernel", [
    (8192, 4096, 60, "none", "tw_gemm_bs_kernel"),    # one step, 64 MB of output, little but stores
    (8192, 4096, 60, "gelu", "tw_gemm_bw_kernel"),
    (8200, 4096, 60, "none", "tw_gemm_bw_kernel"),    # (columns of C off the sectors of memory)
    (10240, 3072, 60, "none", "tw_gemm_bw_kernel"),   # (its workgroups not even)
    (14336, 4096, 60, "none", "tw_gemm_bw_kernel"),   # 112 MB
    (16384, 4096, 60, "relu", "tw_gemm_bs_kernel"),   # 128 MB, columns of C 32 KB apart
    (16384, 4096, 120, "relu", "tw_gemm_bs_kernel"),
    (16320, 4096, 120, "relu", "tw_gemm_bw_kernel"),
    (16384, 4096, 190, "none", "tw_gemm_bw_kernel"),  # three steps
    (8192, 4096, 256, "none", "tw_gemm_bw_kernel"),   # four steps
])
def test_which_weight_stationary_kernel_runs(tw, M, N, kept, act, kernel):
    """The automatic choice between the two (what test_both_weight_stationary_kernels forces runs by itself at these sizes)."""
    K, G = 1024, 128
    tiles = make_tiles(np.random.default_rng(3), K, G, ((kept, G),) * (N // G))
    with tw.Plan.create(K, N, "bf16", tiles, np.zeros((K, N), np.float32)) as plan:
        assert plan.choice(M)["shape"] == tw.SHAPE_BS
        assert plan.kernel_name(M, activation={"none": tw.ACT_NONE, "relu": tw.ACT_RELU, "gelu": tw.ACT_GELU}[act]) == kernel
