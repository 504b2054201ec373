"""GPU parity of the TW GEMM against the CPU oracle, through the C ABI.

Tolerance (stated by the task): max relative error <= 1e-2 for fp16 and <= 2e-2 for
bf16, measured as max |C - C_ref| / max(|C_ref|, 1e-2 * rms(C_ref)) against the
oracle's fp64 dense matmul of the masked weight on the same 16-bit inputs.  Integer
outcomes (which columns are written, untouched sentinels) are checked bit-exactly.
"""
import numpy as np
import pytest

from tests.helpers import from_device_bits, random_tiles, to_device_bits

pytestmark = pytest.mark.gpu

TOL = {"f16": 1e-2, "bf16": 2e-2}
SENTINEL = 0x1234  # 16-bit pattern pre-filled into C


def round_up(v, m):
    return (v + m - 1) // m * m


def run_gemm(tw, oracle, plan, A, dtype, N, alpha=1.0, beta=0.0, C0=None, pruned=0, pad=0):
    """A: fp32 [M,K] -> device K-major 16-bit; returns (C as fp32 [M,N], raw C bits [N,ldc])."""
    import torch
    M, K = A.shape
    lda = round_up(M, 8) + pad
    ldc = round_up(M, 8) + pad
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    Cb = np.full((N, ldc), SENTINEL, np.uint16)
    if C0 is not None:
        Cb[:, :M] = oracle.cast_bits(C0, dtype).reshape(M, N).T
    dA = to_device_bits(At, (K, lda))
    dC = to_device_bits(Cb, (N, ldc))
    plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
              pruned_cols=pruned, stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    bits = from_device_bits(dC)
    return oracle.bits_to_f32(bits[:, :M], dtype).reshape(N, M).T.copy(), bits


def reference(oracle, A, B, tiles, dtype, alpha=1.0, beta=0.0, C0=None):
    Aq, Bq = oracle.quantize(A, dtype), oracle.quantize(B, dtype)
    Cq = None if C0 is None else oracle.quantize(C0, dtype)
    return oracle.tw_gemm_reference(Aq, Bq, tiles, alpha, beta, Cq)


def kept_columns(tiles, N):
    keep = np.zeros(N, bool)
    for t in tiles:
        keep[np.asarray(t["kept_n"], np.int64) + t["col0"]] = True
    return keep


CASES = [
    # M,  K,   N,   G,  k_keep n_keep empty
    (128, 64, 128, 128, 0.5, 1.0, 0),
    (256, 128, 256, 128, 0.25, 1.0, 0),
    (100, 96, 200, 128, 0.3, 0.9, 0),     # ragged M, ragged last tile, K_t not multiples of 32
    (8, 40, 64, 64, 0.5, 0.8, 0),         # tiny M, G = 64 kernel
    (520, 300, 320, 64, 0.2, 0.8, 3),     # G = 64, empty tiles
    (333, 257, 384, 128, 0.25, 0.9, 4),   # M not a multiple of 8
    (1024, 768, 512, 128, 0.25, 1.0, 0),
    (64, 512, 130, 128, 0.1, 0.5, 0),     # last tile 2 columns wide
    (257, 64, 96, 32, 0.5, 0.75, 2),      # G = 32
    (192, 200, 512, 256, 0.3, 0.9, 0),    # tiles wider than one work unit
    (300, 96, 5120, 128, 0.5, 1.0, 7),    # more units than fit the kernel-argument table
    (2048, 64, 4224, 128, 0.6, 0.9, 0),   # several items per workgroup, one 64-row step each
]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("case", CASES)
def test_gemm_matches_oracle(tw, oracle, case, dtype):
    M, K, N, G, kk, nk, empty = case
    rng = np.random.default_rng(hash(case) % (2 ** 31))
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=kk, n_keep=nk, empty_every=empty)
    print("case", case, dtype, flush=True)
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        C, bits = run_gemm(tw, oracle, plan, A, dtype, N, pad=8)
    ref = reference(oracle, A, B, tiles, dtype)
    keep = kept_columns(tiles, N)
    err = oracle.rel_error(C[:, keep], ref[:, keep])
    assert err <= TOL[dtype], err
    # pruned columns and the padding rows beyond M were never written
    assert np.all(bits[~keep, :] == SENTINEL)
    assert np.all(bits[:, M:] == SENTINEL)
    # the reference's own acceptance rule (basic_nn.cu:771-798, err 1e-2) on the kept part
    big = np.abs(ref[:, keep]) > 0.05
    assert oracle.checkout(np.where(big, C[:, keep], 0), np.where(big, ref[:, keep], 0),
                           err=2e-2 if dtype == "bf16" else 1e-2) == 0


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_alpha_beta_and_zero_mode(tw, oracle, dtype):
    rng = np.random.default_rng(21)
    M, K, N, G = 200, 160, 256, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.7)
    keep = kept_columns(tiles, N)
    C0q = oracle.quantize(C0, dtype)
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        # beta != 0: C read only on kept columns, pruned ones untouched (bit-exact)
        C, bits = run_gemm(tw, oracle, plan, A, dtype, N, alpha=0.5, beta=-1.5, C0=C0)
        ref = reference(oracle, A, B, tiles, dtype, 0.5, -1.5, C0)
        assert oracle.rel_error(C[:, keep], ref[:, keep]) <= TOL[dtype]
        assert np.array_equal(C[:, ~keep], C0q[:, ~keep])
        # zero mode, beta == 0: pruned columns become exact zeros
        C, bits = run_gemm(tw, oracle, plan, A, dtype, N, alpha=2.0, C0=C0, pruned=tw.PRUNED_ZERO)
        ref = reference(oracle, A, B, tiles, dtype, 2.0)
        assert oracle.rel_error(C[:, keep], ref[:, keep]) <= TOL[dtype]
        assert np.all(bits[~keep, :M] == 0)
        assert np.all(bits[:, M:] == SENTINEL)
        # zero mode with beta: pruned columns receive beta * C, the full product's value
        C, _ = run_gemm(tw, oracle, plan, A, dtype, N, alpha=1.0, beta=0.5, C0=C0,
                        pruned=tw.PRUNED_ZERO)
        full = oracle.quantize(A, dtype).astype(np.float64) @ oracle.masked_dense_weight(
            oracle.quantize(B, dtype), tiles).astype(np.float64) + 0.5 * C0q
        assert oracle.rel_error(C, full) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_row_major_columns_in_groups_of_four(tw, oracle, dtype):
    """Row-major A and C on a plan whose kept columns are neighbours in C (no column pruned: the
    A-stationary kernel then stores 16-byte pieces of rows) or come in groups of four (element-wise
    stores in the blocks that hold an odd group).  Bit for bit the K-major result with bias and
    ReLU, within tolerance with GELU; ragged M, padding and pruned columns untouched, a C that
    starts 16 bytes into its buffer, a bias that is not 16-byte aligned."""
    import torch
    rng = np.random.default_rng(77)
    M, K, N, G = 203, 320, 512, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = []
    for t in range(N // G):
        quads = np.arange(G // 4) if t % 2 == 0 else np.sort(rng.choice(G // 4, 19, replace=False))
        kept_n = (quads[:, None] * 4 + np.arange(4)).reshape(-1).astype(np.int32)
        kept_k = np.sort(rng.choice(K, K * 2 // 5, replace=False)).astype(np.int32)
        tiles.append(dict(col0=t * G, width=G, kept_k=kept_k, kept_n=kept_n))
    keep = kept_columns(tiles, N)
    Ab = oracle.cast_bits(A, dtype).reshape(M, K)
    d_bias = torch.from_numpy(bias).cuda()
    d_bias1 = torch.from_numpy(np.concatenate([[0.0], bias]).astype(np.float32)).cuda()
    ld8 = round_up(M, 8)
    Ak = np.zeros((K, ld8), np.uint16)
    Ak[:, :M] = Ab.T
    lda = K + 8
    Ar = np.zeros((M, lda), np.uint16)
    Ar[:, :K] = Ab
    pre = 0.75 * reference(oracle, A, B, tiles, dtype) + bias
    refs = {tw.ACT_RELU: np.maximum(pre, 0.0),
            tw.ACT_GELU: 0.5 * pre * (1.0 + np.tanh(np.sqrt(2.0 / np.pi) * (pre + 0.044715 * pre ** 3)))}
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        dAk, dAr = to_device_bits(Ak, Ak.shape), to_device_bits(Ar, Ar.shape)
        for act, ref in refs.items():
            dCk = to_device_bits(np.full((N, ld8), SENTINEL, np.uint16), (N, ld8))
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_AS32)   # (the default for so few rows sums k in four slices)
            try:
                plan.gemm(dAk.data_ptr(), dCk.data_ptr(), M, lda=ld8, ldc=ld8, alpha=0.75,
                          bias_ptr=d_bias.data_ptr(), activation=act)
            finally:
                tw.set_option(tw.OPT_SHAPE, -1)
            torch.cuda.synchronize()
            want = from_device_bits(dCk)[:, :M].T
            want_f = oracle.bits_to_f32(np.ascontiguousarray(want), dtype).reshape(M, N)
            assert oracle.rel_error(want_f[:, keep], ref[:, keep]) <= TOL[dtype]
            # 8-byte stores; a bias that is not 16-byte aligned: element-wise stores
            for ldc, shift, bias_shift in ((N + 8, 0, 0), (N + 16, 8, 0), (N + 8, 0, 1)):
                full = torch.full((M * ldc + 16,), SENTINEL, dtype=torch.int16, device="cuda")
                plan.gemm(dAr.data_ptr(), full.data_ptr() + 2 * shift, M, lda=lda, ldc=ldc, alpha=0.75,
                          a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR,
                          bias_ptr=(d_bias1.data_ptr() + 4) if bias_shift else d_bias.data_ptr(),
                          activation=act)
                torch.cuda.synchronize()
                flat = full.cpu().numpy().view(np.uint16)
                assert np.all(flat[:shift] == SENTINEL) and np.all(flat[shift + M * ldc:] == SENTINEL)
                got = flat[shift:shift + M * ldc].reshape(M, ldc)
                assert np.all(got[:, N:] == SENTINEL)
                assert np.all(got[:, :N][:, ~keep] == SENTINEL)
                if act == tw.ACT_RELU:      # the same arithmetic in every kernel: the same bits
                    assert np.array_equal(got[:, :N][:, keep], want[:, keep])
                else:
                    got_f = oracle.bits_to_f32(np.ascontiguousarray(got[:, :N]), dtype).reshape(M, N)
                    assert oracle.rel_error(got_f[:, keep], ref[:, keep]) <= TOL[dtype]
                    assert oracle.rel_error(got_f[:, keep], want_f[:, keep]) <= 0.5 * TOL[dtype]


@pytest.mark.parametrize("staged", [False, True])
@pytest.mark.parametrize("a_layout,c_layout", [(1, 1), (1, 0), (0, 1)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_row_major_layouts(tw, oracle, a_layout, c_layout, dtype, staged):
    """Row-major A[M,K] (lda >= K) and/or C[M,N] (ldc >= N): through the layout-generic kernel, and
    staged through K-major copies in a caller's workspace (tw_gemm_staged).  Ragged sizes: M, K
    and N are no multiples of 8, the leading dimensions leave padding that must stay untouched."""
    import torch
    rng = np.random.default_rng(31 + 2 * a_layout + c_layout)
    M, K, N, G = 203, 150, 330, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.8, empty_every=3)
    keep = kept_columns(tiles, N)
    Ab, Cb = oracle.cast_bits(A, dtype).reshape(M, K), oracle.cast_bits(C0, dtype).reshape(M, N)
    if a_layout == tw.ROWMAJOR:
        lda = round_up(K, 8) + 8
        Ah = np.zeros((M, lda), np.uint16)
        Ah[:, :K] = Ab
    else:
        lda = round_up(M, 8)
        Ah = np.zeros((K, lda), np.uint16)
        Ah[:, :M] = Ab.T
    for alpha, beta, pruned in ((1.0, 0.0, tw.PRUNED_UNTOUCHED), (0.5, 2.0, tw.PRUNED_ZERO)):
        if c_layout == tw.ROWMAJOR:
            ldc = round_up(N, 8) + 8
            Ch = np.full((M, ldc), SENTINEL, np.uint16)
            Ch[:, :N] = Cb
        else:
            ldc = round_up(M, 8)
            Ch = np.full((N, ldc), SENTINEL, np.uint16)
            Ch[:, :M] = Cb.T
        dA, dC = to_device_bits(Ah, Ah.shape), to_device_bits(Ch, Ch.shape)
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            kw = {}
            if staged:
                nbytes = plan.staged_workspace(M, a_layout, c_layout)
                assert nbytes == 2 * round_up(M, 64) * (K * (a_layout == tw.ROWMAJOR) +
                                                        N * (c_layout == tw.ROWMAJOR))
                ws = torch.full((nbytes // 2 + 64,), 0x7bcd, dtype=torch.int16, device="cuda")
                kw = dict(workspace_ptr=ws.data_ptr(), workspace_bytes=nbytes)
                # (beta != 0: a workspace is asked for whatever the layouts are; with beta == 0 and this short K two
                # row-major operands need none.  At these sizes the few-rows kernel takes two row-major operands as
                # they are all the same; both staged: test_gemm_both_row_major_operands_staged)
                with pytest.raises(tw.TwError) as e:
                    plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, beta=1.0, a_layout=a_layout,
                              c_layout=c_layout, workspace_ptr=ws.data_ptr(), workspace_bytes=nbytes - 2)
                assert e.value.status == tw.ERR_BUFFER
            plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
                      a_layout=a_layout, c_layout=c_layout, pruned_cols=pruned, **kw)
            torch.cuda.synchronize()
            if staged:
                assert torch.all(ws[nbytes // 2:] == 0x7bcd)   # nothing beyond the stated size
                # the staged path is the K-major kernel on transposed copies: bit for bit what
                # that kernel gives on K-major operands
                Ak = np.zeros((K, round_up(M, 8)), np.uint16)
                Ak[:, :M] = Ab.T
                Ck = np.full((N, round_up(M, 8)), SENTINEL, np.uint16)
                Ck[:, :M] = Cb.T
                dAk, dCk = to_device_bits(Ak, Ak.shape), to_device_bits(Ck, Ck.shape)
                plan.gemm(dAk.data_ptr(), dCk.data_ptr(), M, lda=round_up(M, 8), ldc=round_up(M, 8),
                          alpha=alpha, beta=beta, pruned_cols=pruned)
                torch.cuda.synchronize()
                want = from_device_bits(dCk)[:, :M].T
                have = from_device_bits(dC)
                have = have[:, :N] if c_layout == tw.ROWMAJOR else have[:, :M].T
                assert np.array_equal(np.ascontiguousarray(have), np.ascontiguousarray(want))
        out = from_device_bits(dC)
        got = out[:, :N] if c_layout == tw.ROWMAJOR else out[:, :M].T
        pad = out[:, N:] if c_layout == tw.ROWMAJOR else out[:, M:]
        assert np.all(pad == SENTINEL)
        Cf = oracle.bits_to_f32(np.ascontiguousarray(got), dtype).reshape(M, N)
        ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
        assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
        if pruned == tw.PRUNED_UNTOUCHED:
            assert np.array_equal(np.ascontiguousarray(got)[:, ~keep], Cb[:, ~keep])
        else:
            expect = oracle.cast_bits(beta * oracle.quantize(C0, dtype)[:, ~keep], dtype)
            assert np.array_equal(np.ascontiguousarray(got)[:, ~keep], expect.reshape(M, -1))


@pytest.mark.parametrize("M,K,N", [(203, 150, 330), (100, 2200, 200)])     # a panel of A fits LDS, or does not
@pytest.mark.parametrize("alpha,beta,pruned", [(1.0, 0.0, 0), (0.5, 2.0, 1)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_both_row_major_operands_staged(tw, oracle, dtype, alpha, beta, pruned, M, K, N):
    """Row-major A and C where no kernel takes them directly (a streaming shape is forced): tw_gemm_staged
    turns both through one workspace, A in front and C's old values behind it, and gives the bits of the same
    shape on K-major operands; tw_gemm_ex takes the layout-generic kernel.  (K 150 with beta == 0 is a
    panel that fits: taken directly whatever shape is forced.)"""
    import torch
    rng = np.random.default_rng(37)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    tiles = random_tiles(rng, K, N, 128, k_keep=0.4, n_keep=0.8)
    keep = kept_columns(tiles, N)
    Ab, Cb = oracle.cast_bits(A, dtype).reshape(M, K), oracle.cast_bits(C0, dtype).reshape(M, N)
    lda, ldc, ldm = round_up(K, 8) + 8, round_up(N, 8) + 8, round_up(M, 8)
    Ah, Ch = np.zeros((M, lda), np.uint16), np.full((M, ldc), SENTINEL, np.uint16)
    Ah[:, :K], Ch[:, :N] = Ab, Cb
    Ak, Ck = np.zeros((K, ldm), np.uint16), np.full((N, ldm), SENTINEL, np.uint16)
    Ak[:, :M], Ck[:, :M] = Ab.T, Cb.T
    dA, dAk, dCk = (to_device_bits(x, x.shape) for x in (Ah, Ak, Ck))
    direct = beta == 0.0 and K == 150
    ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
    tw.set_option(tw.OPT_SHAPE, tw.SHAPE_128x128)
    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            nbytes = plan.staged_workspace(M, tw.ROWMAJOR, tw.ROWMAJOR)
            assert nbytes == 2 * round_up(M, 64) * (K + N)
            ws = torch.full((nbytes // 2 + 64,), 0x7bcd, dtype=torch.int16, device="cuda")
            kw = dict(alpha=alpha, beta=beta, pruned_cols=pruned)
            row = dict(lda=lda, ldc=ldc, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR)
            got = {}
            for name, extra in (("staged", dict(workspace_ptr=ws.data_ptr(), workspace_bytes=nbytes)), ("generic", {})):
                dC = to_device_bits(Ch, Ch.shape)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, **kw, **row, **extra)
                torch.cuda.synchronize()
                got[name] = from_device_bits(dC)
            plan.gemm(dAk.data_ptr(), dCk.data_ptr(), M, lda=ldm, ldc=ldm, **kw)
            torch.cuda.synchronize()
            want = from_device_bits(dCk)[:, :M].T
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
    assert torch.all(ws[nbytes // 2:] == 0x7bcd)                      # nothing beyond the stated size
    assert torch.all(ws[:nbytes // 2] == 0x7bcd) == direct            # the workspace was used, or not needed
    for name, out in got.items():
        assert np.all(out[:, N:] == SENTINEL)
        Cf = oracle.bits_to_f32(np.ascontiguousarray(out[:, :N]), dtype).reshape(M, N)
        assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype], name
        assert np.array_equal(np.ascontiguousarray(out[:, :N])[:, ~keep], np.ascontiguousarray(want)[:, ~keep]), name
    if not direct:
        assert np.array_equal(got["staged"][:, :N], want)


def test_gemm_degenerate_plans(tw, oracle):
    rng = np.random.default_rng(22)
    M, K, N, G = 96, 64, 256, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    e = np.zeros(0, np.int32)
    # tile 0 keeps columns but no K row -> zeros there; tile 1 keeps no column -> untouched
    tiles = [dict(col0=0, width=128, kept_k=e, kept_n=np.arange(0, 128, 3, dtype=np.int32)),
             dict(col0=128, width=128, kept_k=np.arange(K, dtype=np.int32), kept_n=e)]
    with tw.Plan.create(K, N, "f16", tiles, B) as plan:
        assert plan.info()["empty_tiles"] == 2
        C, bits = run_gemm(tw, oracle, plan, A, "f16", N)
        keep = kept_columns(tiles, N)
        assert np.all(bits[keep, :M] == 0) and np.all(bits[~keep, :] == SENTINEL)
        # M == 0 is a no-op
        plan.gemm(0, 0, 0)
    # identity weight: C is the gathered A columns, exactly
    K = N = 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    kk = np.sort(rng.choice(K, 37, replace=False)).astype(np.int32)
    one = [dict(col0=0, width=N, kept_k=kk, kept_n=np.arange(N, dtype=np.int32))]
    with tw.Plan.create(K, N, "f16", one, np.eye(K, dtype=np.float32)) as plan:
        C, _ = run_gemm(tw, oracle, plan, A, "f16", N)
    expect = np.zeros((M, N), np.float32)
    expect[:, kk] = oracle.quantize(A, "f16")[:, kk]
    assert np.array_equal(C, expect)


def test_dense_plan_equals_plain_gemm(tw, oracle):
    import torch
    rng = np.random.default_rng(23)
    M, K, N, G = 512, 384, 640, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    with tw.Plan.dense(K, N, G, "f16", B) as plan:
        C, _ = run_gemm(tw, oracle, plan, A, "f16", N)
    Aq, Bq = oracle.quantize(A, "f16"), oracle.quantize(B, "f16")
    assert oracle.rel_error(C, Aq.astype(np.float64) @ Bq.astype(np.float64)) <= TOL["f16"]
    # a library routine on the same inputs (hipBLASLt/rocBLAS through torch)
    lib = (torch.from_numpy(Aq).cuda().half() @ torch.from_numpy(Bq).cuda().half()).float().cpu().numpy()
    assert oracle.rel_error(C, lib) <= TOL["f16"]


def test_fused_equals_gather_dense_scatter_bitwise(tw, oracle):
    """The reference's first self-check (basic_nn.cu:1081, tolerance 1e-10 = exact): the
    fused masked GEMM equals gather rows -> dense GEMM on the compact tile -> scatter,
    run through the engine's own kernel and its deleteRow / insertRow kernels."""
    import torch
    rng = np.random.default_rng(24)
    M, K, N, G, dtype = 264, 320, 384, 128, "f16"
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.3, n_keep=0.8)
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        _, fused = run_gemm(tw, oracle, plan, A, dtype, N)
    At = oracle.cast_bits(A, dtype).reshape(M, K).T.copy()
    dA = to_device_bits(At, (K, M))
    out = np.full((N, M), SENTINEL, np.uint16)
    for t in tiles:
        kt, nt = len(t["kept_k"]), len(t["kept_n"])
        rel_k = torch.from_numpy(t["kept_k"] - np.arange(kt, dtype=np.int32)).cuda()
        rel_n = torch.from_numpy(t["kept_n"] - np.arange(nt, dtype=np.int32)).cuda()
        dA2 = torch.zeros((kt, M), dtype=torch.int16, device="cuda")
        tw.delete_row(dA.data_ptr(), dA2.data_ptr(), kt, M, rel_k.data_ptr())
        comp = B[np.ix_(t["kept_k"], t["kept_n"] + t["col0"])]
        dC2 = torch.zeros((nt, M), dtype=torch.int16, device="cuda")
        with tw.Plan.dense(kt, nt, max(nt, 1), dtype, comp) as dense:
            dense.gemm(dA2.data_ptr(), dC2.data_ptr(), M)
            torch.cuda.synchronize()
        dCt = to_device_bits(out[t["col0"]:t["col0"] + t["width"]], (t["width"], M))
        tw.insert_row(dCt.data_ptr(), dC2.data_ptr(), nt, M, rel_n.data_ptr())
        torch.cuda.synchronize()
        out[t["col0"]:t["col0"] + t["width"]] = from_device_bits(dCt)
    assert np.array_equal(fused[:, :M], out)


def test_tile_order_does_not_change_a_bit(tw, oracle):
    """Work-queue order must not matter: the same tiles with kept-K counts arranged so
    that the queue sorts them differently give bit-identical columns."""
    rng = np.random.default_rng(25)
    M, K, N, G, dtype = 300, 256, 512, 128, "f16"
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.3, n_keep=0.9)
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        _, base = run_gemm(tw, oracle, plan, A, dtype, N)
    # reverse the column-tile order of the weight (and of the plan): each tile's columns
    # must come out identical, at their new position
    perm = list(reversed(range(len(tiles))))
    B2 = np.concatenate([B[:, tiles[i]["col0"]:tiles[i]["col0"] + G] for i in perm], axis=1)
    tiles2 = [dict(col0=j * G, width=G, kept_k=tiles[i]["kept_k"], kept_n=tiles[i]["kept_n"])
              for j, i in enumerate(perm)]
    with tw.Plan.create(K, N, dtype, tiles2, B2) as plan:
        _, moved = run_gemm(tw, oracle, plan, A, dtype, N)
    for j, i in enumerate(perm):
        assert np.array_equal(moved[j * G:(j + 1) * G], base[i * G:(i + 1) * G])


def test_repeated_launches_and_slot_reuse(tw, oracle):
    """More launches than ticket slots on one plan: every launch must see a re-armed queue."""
    import torch
    rng = np.random.default_rng(26)
    M, K, N, G, dtype = 136, 96, 256, 128, "f16"
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.5, n_keep=0.9)
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        _, first = run_gemm(tw, oracle, plan, A, dtype, N)
        At = oracle.cast_bits(A, dtype).reshape(M, K).T.copy()
        dA = to_device_bits(At, (K, M))
        dC = torch.zeros((N, M), dtype=torch.int16, device="cuda")
        for _ in range(600):
            plan.gemm(dA.data_ptr(), dC.data_ptr(), M,
                      stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        keep = kept_columns(tiles, N)
        assert np.array_equal(from_device_bits(dC)[keep], first[keep, :M])


def test_plan_reset_leaves_results_unchanged(tw, oracle):
    """tw_plan_reset between launches (the call that re-arms every ticket slot after an aborted
    launch): the launches after it give the bits of the launches before it."""
    import torch
    rng = np.random.default_rng(28)
    M, K, N, G, dtype = 300, 192, 640, 128, "f16"
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.5, n_keep=0.9)
    stream = torch.cuda.current_stream().cuda_stream
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        _, first = run_gemm(tw, oracle, plan, A, dtype, N)
        ld = (M + 7) // 8 * 8
        At = np.zeros((K, ld), np.uint16)
        At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
        dA = to_device_bits(At, (K, ld))
        keep = kept_columns(tiles, N)
        for _ in range(3):
            plan.reset(stream)
            dC = torch.zeros((N, ld), dtype=torch.int16, device="cuda")
            for _ in range(5):
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=ld, ldc=ld, stream=stream)
            torch.cuda.synchronize()
            assert np.array_equal(from_device_bits(dC)[keep, :M], first[keep, :M])
    assert tw.lib().tw_plan_reset(None, None) == tw.ERR_NULL


def test_queue_is_rearmed_between_launches_of_different_sizes(tw, oracle):
    """Launches with few items (one per workgroup), with several rounds of items per workgroup,
    and with items that have no step or only fill zeros alternate on one plan, through every
    ticket slot more than once: each launch re-arms the queue for the next, whatever its grid
    was, so every result repeats bit for bit."""
    import torch
    rng = np.random.default_rng(27)
    K, N, G, dtype = 320, 1536, 128, "bf16"
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.85, empty_every=5)
    Ms = (8, 520, 33000)                  # 12 items; 36 items; 129 row blocks x 12 units
    stream = torch.cuda.current_stream().cuda_stream
    with tw.Plan.create(K, N, dtype, tiles, B) as plan:
        dA, dC, want = {}, {}, {}
        for M in Ms:
            ld = (M + 7) // 8 * 8
            g = torch.Generator(device="cuda")
            g.manual_seed(M)
            dA[M] = torch.randn((K, ld), generator=g, device="cuda").to(torch.bfloat16)
            dC[M] = torch.zeros((N, ld), dtype=torch.bfloat16, device="cuda")
            plan.gemm(dA[M].data_ptr(), dC[M].data_ptr(), M, lda=ld, ldc=ld, stream=stream,
                      pruned_cols=tw.PRUNED_ZERO)
            torch.cuda.synchronize()
            want[M] = dC[M].clone()
            ref = (dA[M][:, :M].float().T.cpu().numpy() @
                   (oracle.quantize(B, dtype) * oracle.plan_mask(K, N, tiles)))
            got = dC[M][:, :M].float().T.cpu().numpy()
            assert oracle.rel_error(got, ref) <= TOL[dtype], M
        print("re-arm over mixed sizes", Ms, flush=True)
        for i in range(3 * 256 + 5):
            M = Ms[i % 3] if i % 7 else Ms[2 - i % 3]
            ld = (M + 7) // 8 * 8
            dC[M].fill_(1.0)
            plan.gemm(dA[M].data_ptr(), dC[M].data_ptr(), M, lda=ld, ldc=ld, stream=stream,
                      pruned_cols=tw.PRUNED_ZERO)
            if i % 64 == 63 or i > 3 * 256:
                torch.cuda.synchronize()
                assert torch.equal(dC[M][:, :M], want[M][:, :M]), (i, M)


def test_gemm_argument_errors(tw):
    import torch
    K, N, M = 64, 128, 64
    with tw.Plan.dense(K, N, 128, "f16", np.zeros((K, N), np.float32)) as plan:
        a = torch.zeros((K, M), dtype=torch.int16, device="cuda")
        c = torch.zeros((N, M), dtype=torch.int16, device="cuda")
        for kwargs, status in ((dict(lda=M - 8), tw.ERR_SHAPE), (dict(ldc=M + 4), tw.ERR_ALIGNMENT),
                               (dict(a_layout=5), tw.ERR_LAYOUT), (dict(pruned_cols=3), tw.ERR_LAYOUT)):
            with pytest.raises(tw.TwError) as e:
                plan.gemm(a.data_ptr(), c.data_ptr(), M, **kwargs)
            assert e.value.status == status
        with pytest.raises(tw.TwError) as e:
            plan.gemm(a.data_ptr() + 2, c.data_ptr(), M)
        assert e.value.status == tw.ERR_ALIGNMENT
        with pytest.raises(tw.TwError) as e:
            plan.gemm(0, c.data_ptr(), M)
        assert e.value.status == tw.ERR_NULL
        with pytest.raises(tw.TwError) as e:
            plan.gemm(a.data_ptr(), c.data_ptr(), -1)
        assert e.value.status == tw.ERR_SHAPE


def test_stream_gemm_nn_drop_in(tw, oracle):
    """The reference's own problem (`test_basic_nn 64 768 256 384 128`, its rand() stream)
    driven through the Stream_Gemm_NN-shaped entry point with the reference's operands."""
    import torch
    M, N, K, Np, Kp = 64, 768, 256, 384, 128
    A, B, tiles, part = oracle.ref_compat_problem(M, N, K, Np, Kp)
    dtype = "f16"
    dA = to_device_bits(oracle.cast_bits(A, dtype).reshape(M, K).T.copy(), (K, M))
    dB = to_device_bits(oracle.cast_bits(oracle.stream_weight(B, tiles), dtype), (K * N,))
    dC = torch.zeros((N, M), dtype=torch.int16, device="cuda")
    mk = [torch.from_numpy(t["mask_k"]).cuda() for t in tiles]
    mn = [torch.from_numpy(t["mask_n"]).cuda() for t in tiles]
    tw.stream_gemm_nn(M, N, K, dtype, 1.0, dA.data_ptr(), dB.data_ptr(), 0.0, dC.data_ptr(),
                      part["N_cal"], part["K_cal"], [x.data_ptr() for x in mn],
                      [x.data_ptr() for x in mk], part["off_B"], part["off_C"])
    C = oracle.bits_to_f32(from_device_bits(dC), dtype).reshape(N, M).T
    ref = reference(oracle, A, B, tiles, dtype)
    assert oracle.rel_error(C, ref) <= TOL[dtype]
    # and a plan built from those operands exports the same lists and weight bits
    with tw.Plan.from_stream_operands(M, N, K, dtype, dB.data_ptr(), part["N_cal"], part["K_cal"],
                                      [x.data_ptr() for x in mn], [x.data_ptr() for x in mk],
                                      part["off_B"], part["off_C"]) as plan:
        got, Bs = plan.export()
        for g, t in zip(got, tiles):
            assert np.array_equal(g["kept_k"], t["kept_k"]) and np.array_equal(g["mask_n"], t["mask_n"])
        assert np.array_equal(Bs, from_device_bits(dB))


@pytest.mark.parametrize("forced", ["auto", "streaming"])
def test_graph_capture_replays_bitwise(tw, oracle, forced):
    """tw_gemm allocates nothing, clears nothing from the host and re-arms its work queue inside
    the kernel, so a sequence of launches can be captured into a HIP graph; every replay (with
    eager launches and synchronisations in between) gives the eager result bit for bit.  Once with
    the kernel the launch picks by itself (none that uses the queue at this size) and once with a
    streaming kernel forced, whose recorded launches keep a ticket slot of the plan's captured
    range across the replays and re-arm it each time."""
    import torch
    rng = np.random.default_rng(77)
    M, K, N, G = 384, 256, 512, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.9)
    At = np.ascontiguousarray(oracle.cast_bits(A, "f16").reshape(M, K).T)
    dA = to_device_bits(At, At.shape)
    dH = torch.zeros((N, M), dtype=torch.int16, device="cuda")
    dC = torch.zeros((N, M), dtype=torch.int16, device="cuda")
    s = torch.cuda.Stream()
    try:
        if forced == "streaming":
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_128x64)
            tw.set_option(tw.OPT_PIECE, 64)
            tw.set_option(tw.OPT_XCD_QUEUES, 1)
        with tw.Plan.create(K, N, "f16", tiles, B) as plan:
            if forced == "streaming":
                assert plan.choice(M)["shape"] == tw.SHAPE_128x64

            def chain():
                # two dependent launches: C = A (B.mask), then C += 0.5 * A (B.mask) on top of it
                plan.gemm(dA.data_ptr(), dH.data_ptr(), M, pruned_cols=tw.PRUNED_ZERO, stream=s.cuda_stream)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, alpha=0.5, beta=0.0, pruned_cols=tw.PRUNED_ZERO,
                          stream=s.cuda_stream)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, alpha=1.0, beta=1.0, stream=s.cuda_stream)
            with torch.cuda.stream(s):
                print("graph capture", forced, flush=True)
                chain()
                s.synchronize()
                want_h, want_c = dH.clone(), dC.clone()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=s):
                    chain()
                for rep in range(4):
                    dH.fill_(0x1234)
                    dC.fill_(0x1234)
                    plan.gemm(dA.data_ptr(), dH.data_ptr(), M, stream=s.cuda_stream)   # eager work between replays
                    s.synchronize()
                    g.replay()
                    s.synchronize()
                    assert torch.equal(dH, want_h) and torch.equal(dC, want_c), rep
    finally:
        for opt in (tw.OPT_SHAPE, tw.OPT_PIECE, tw.OPT_XCD_QUEUES):
            tw.set_option(opt, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_every_kernel_shape_agrees(tw, oracle, dtype):
    """The launch picks a kernel shape, the width of a unit piece and the queue layout from the
    plan and M; tw_set_option forces each combination a plan can run with in turn: all match the
    oracle, and each repeats itself bit for bit."""
    rng = np.random.default_rng(88)
    W, S1, S2, S3, S4, S5 = (tw.SHAPE_WIDE, tw.SHAPE_128x128, tw.SHAPE_512x64, tw.SHAPE_128x64,
                             tw.SHAPE_256x128, tw.SHAPE_128x32)
    A6, A3, SK, BS, S6 = tw.SHAPE_AS64, tw.SHAPE_AS32, tw.SHAPE_SKINNY, tw.SHAPE_BS, tw.SHAPE_256x64
    cases = (
        (600, 320, 384, 128, ((W, -1), (S1, -1), (S4, -1), (S3, 64), (S5, 32), (S1, 64), (S4, 32),
                              (A6, -1), (A3, -1), (SK, -1), (BS, -1))),
        (1100, 200, 256, 64, ((S2, -1), (S3, -1), (S5, 32), (S1, -1), (S4, -1), (W, -1), (A6, -1),
                              (A3, -1), (SK, -1), (BS, -1), (S6, -1), (S6, 32))),
        (2500, 130, 96, 32, ((S5, -1), (S3, -1), (S2, -1), (A6, -1), (A3, -1), (SK, -1), (BS, -1), (S6, -1), (S6, 32))),
    )
    try:
        for (M, K, N, G, combos) in cases:
            A = rng.standard_normal((M, K)).astype(np.float32)
            B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
            tiles = random_tiles(rng, K, N, G, k_keep=0.45, n_keep=0.85)
            ref = reference(oracle, A, B, tiles, dtype)
            keep = kept_columns(tiles, N)
            with tw.Plan.create(K, N, dtype, tiles, B) as plan:
                for shape, piece in combos:
                    for xcd in (1, 0, 2):
                        tw.set_option(tw.OPT_SHAPE, shape)
                        tw.set_option(tw.OPT_PIECE, piece)
                        tw.set_option(tw.OPT_XCD_QUEUES, xcd)
                        print("shape", shape, "piece", piece, "xcd", xcd, M, K, N, G, dtype, flush=True)
                        C1, bits1 = run_gemm(tw, oracle, plan, A, dtype, N)
                        C2, bits2 = run_gemm(tw, oracle, plan, A, dtype, N)
                        assert oracle.rel_error(C1[:, keep], ref[:, keep]) <= TOL[dtype], (shape, piece)
                        assert np.array_equal(bits1, bits2), (shape, piece)
                        if shape in (S4, S6):
                            # the 256-row kernels load straight into LDS by default; their
                            # register-staged form gives the same bits
                            tw.set_option(tw.OPT_LDS_DMA, 0)
                            C3, bits3 = run_gemm(tw, oracle, plan, A, dtype, N)
                            tw.set_option(tw.OPT_LDS_DMA, -1)
                            assert np.array_equal(bits1, bits3), (shape, piece, "register-staged")
    finally:
        for opt in (tw.OPT_SHAPE, tw.OPT_PIECE, tw.OPT_XCD_QUEUES, tw.OPT_LDS_DMA):
            tw.set_option(opt, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_a_stationary_shapes(tw, oracle, dtype):
    """The A-stationary kernels (a panel of A resident in LDS, kept rows gathered inside LDS) are
    forced with tw_set_option here.  Tiles from no kept row to all of them (one to nine segments of
    two steps), ragged M, bias + activation, filled pruned columns: bit for bit what the streaming
    256 x 128 kernel gives, and within tolerance of the oracle.  With beta != 0 (C is read) the
    forced shape does not apply and the launch takes the default kernel (for these few rows the
    skinny one, whose sums run in slices: within half the tolerance)."""
    rng = np.random.default_rng(4321)
    M, K, N, G = 333, 1040, 640, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = []
    for t, (kt, nt) in enumerate(((1040, 128), (64, 100), (0, 128), (333, 128), (700, 7))):
        tiles.append(dict(col0=t * G, width=G,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(G, size=nt, replace=False)).astype(np.int32)))
    keep = kept_columns(tiles, N)
    import torch
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = round_up(M, 8)
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)

    def launch(plan, shape, alpha, beta, pruned, with_bias, act):
        Cb = np.full((N, ldc), SENTINEL, np.uint16)
        Cb[:, :M] = oracle.cast_bits(C0, dtype).reshape(M, N).T
        dC = to_device_bits(Cb, Cb.shape)
        tw.set_option(tw.OPT_SHAPE, shape)
        print("a-stationary test: shape", shape, alpha, beta, pruned, with_bias, act, dtype, flush=True)
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
                  pruned_cols=pruned, bias_ptr=dbias.data_ptr() if with_bias else None, activation=act,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, beta, pruned, with_bias, act) in (
                    (1.0, 0.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                    (0.5, 0.0, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                    (1.0, 0.0, tw.PRUNED_ZERO, True, tw.ACT_GELU),
                    (2.0, 0.75, tw.PRUNED_ZERO, False, tw.ACT_NONE)):
                want = launch(plan, tw.SHAPE_256x128, alpha, beta, pruned, with_bias, act)
                for shape in (tw.SHAPE_AS64, tw.SHAPE_AS32):
                    got = launch(plan, shape, alpha, beta, pruned, with_bias, act)
                    if act == tw.ACT_GELU or beta != 0.0:
                        # the two kernels evaluate the polynomial inside GELU in loops of their
                        # own; the compiler fuses their multiply-adds differently: last-bit ties
                        a = oracle.bits_to_f32(got[:, :M], dtype)
                        b = oracle.bits_to_f32(want[:, :M], dtype)
                        assert oracle.rel_error(a, b) <= 0.5 * TOL[dtype]
                        assert np.array_equal(got[:, M:], want[:, M:])
                    else:
                        assert np.array_equal(got, want), (shape, alpha, beta, pruned, with_bias, act)
                if not with_bias and act == tw.ACT_NONE:
                    Cf = oracle.bits_to_f32(want[:, :M], dtype).reshape(N, M).T
                    ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
                    assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_row_blocks_sized_per_tile(tw, oracle, dtype):
    """A launch whose items would not fill the chip once gives the tiles with more kept rows lower
    row blocks (multiples of 64 rows).  Tiles of 40 to 900 kept rows, one without any, ragged M,
    pruned columns filled, bias + activation, beta: every streaming shape gives the same bits with
    TW_OPT_BALANCE 0 and 1 and stays within tolerance of the oracle; nothing is written past M."""
    import torch
    rng = np.random.default_rng(8086)
    M, K, N, G = 5003, 1000, 640, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = []
    for t, (kt, nt) in enumerate(((900, 128), (40, 100), (0, 128), (333, 128), (520, 77))):
        tiles.append(dict(col0=t * G, width=G,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(G, size=nt, replace=False)).astype(np.int32)))
    keep = kept_columns(tiles, N)
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = round_up(M, 8) + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)

    def launch(plan, shape, balance, alpha, beta, pruned, with_bias, act):
        Cb = np.full((N, ldc), SENTINEL, np.uint16)
        Cb[:, :M] = oracle.cast_bits(C0, dtype).reshape(M, N).T
        dC = to_device_bits(Cb, Cb.shape)
        tw.set_option(tw.OPT_SHAPE, shape)
        tw.set_option(tw.OPT_BALANCE, balance)
        print("row blocks per tile: shape", shape, balance, alpha, beta, pruned, with_bias, act, dtype, flush=True)
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
                  pruned_cols=pruned, bias_ptr=dbias.data_ptr() if with_bias else None, activation=act,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, beta, pruned, with_bias, act) in (
                    (1.0, 0.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                    (0.5, 0.0, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                    (2.0, 0.75, tw.PRUNED_ZERO, False, tw.ACT_NONE)):
                for shape in (tw.SHAPE_256x128, tw.SHAPE_128x128):
                    want = launch(plan, shape, 0, alpha, beta, pruned, with_bias, act)
                    got = launch(plan, shape, 1, alpha, beta, pruned, with_bias, act)
                    assert np.array_equal(got, want), (shape, alpha, beta, pruned, with_bias, act)
                    assert (got[:, M:] == SENTINEL).all()
                    if not with_bias and act == tw.ACT_NONE:
                        Cf = oracle.bits_to_f32(got[:, :M], dtype).reshape(N, M).T
                        ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
                        assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
        tw.set_option(tw.OPT_BALANCE, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("shape_bn", [128, 64])
def test_streaming_kernel_several_items_per_workgroup(tw, oracle, dtype, shape_bn):
    """The 256-row streaming kernels with more items than workgroups, so that every workgroup runs
    several one after the other: the first steps of the next item are loaded over the epilogue of
    the current one, and a full C tile (every column kept, 256 rows) is stored by the moving waves
    during the next item's first time slot.  Tiles of 1 to 7 steps, one without kept rows, full
    and partly kept columns, a ragged last row block: the same bits as the register-staged form of
    the kernel (TW_OPT_LDS_DMA = 0) and as a second launch, within tolerance of the oracle, with
    bias + activation and filled pruned columns as well."""
    import torch
    rng = np.random.default_rng(31337 + shape_bn)
    G = shape_bn
    n_tiles = 40 if G == 128 else 72
    M, K, N = 2048 + 256 * 5 + 77, 448, n_tiles * G          # 14 row blocks, the last one ragged
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = []
    for t in range(n_tiles):
        kt = (64, 128, 200, 448, 0, 130, 70, 256)[t % 8]
        nt = G if t % 3 else int(G * 0.8)
        tiles.append(dict(col0=t * G, width=G,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(G, size=nt, replace=False)).astype(np.int32)))
    keep = kept_columns(tiles, N)
    ref = reference(oracle, A, B, tiles, dtype)
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = round_up(M, 8)
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)
    shape = tw.SHAPE_256x128 if G == 128 else tw.SHAPE_256x64

    def launch(plan, dma, pruned, with_bias, act):
        dC = to_device_bits(np.full((N, ldc), SENTINEL, np.uint16), (N, ldc))
        tw.set_option(tw.OPT_LDS_DMA, dma)
        print("several items per workgroup:", G, dma, pruned, with_bias, act, dtype, flush=True)
        assert plan.choice(M, lda, ldc)["shape"] == shape
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, pruned_cols=pruned,
                  bias_ptr=dbias.data_ptr() if with_bias else None, activation=act,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    try:
        tw.set_option(tw.OPT_SHAPE, shape)
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (pruned, with_bias, act) in ((tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                                             (tw.PRUNED_ZERO, True, tw.ACT_RELU)):
                want = launch(plan, 0, pruned, with_bias, act)
                for rep in range(2):
                    got = launch(plan, 1, pruned, with_bias, act)
                    assert np.array_equal(got, want), (rep, pruned, with_bias, act)
                assert (want[:, M:] == SENTINEL).all()
                if not with_bias:
                    Cf = oracle.bits_to_f32(want[:, :M], dtype).reshape(N, M).T
                    assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
                    assert (want[~keep] == SENTINEL).all()
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
        tw.set_option(tw.OPT_LDS_DMA, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_256x64_shape_epilogues(tw, oracle, dtype):
    """The 256 x 64 streaming shape (64-wide tiles of plans with few items) with every epilogue:
    alpha / beta, bias + activation, filled pruned columns, both queue layouts and both piece
    widths it takes: bit for bit what the 128 x 64 shape gives (same step order over k, same
    epilogue code), within tolerance of the oracle, nothing written past M."""
    import torch
    rng = np.random.default_rng(6464)
    M, K, N, G = 777, 300, 320, 64
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.8)
    keep = kept_columns(tiles, N)
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = round_up(M, 8) + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)

    def launch(plan, shape, piece, xcd, alpha, beta, pruned, with_bias, act):
        Cb = np.full((N, ldc), SENTINEL, np.uint16)
        Cb[:, :M] = oracle.cast_bits(C0, dtype).reshape(M, N).T
        dC = to_device_bits(Cb, Cb.shape)
        tw.set_option(tw.OPT_SHAPE, shape)
        tw.set_option(tw.OPT_PIECE, piece)
        tw.set_option(tw.OPT_XCD_QUEUES, xcd)
        print("256x64 test: shape", shape, piece, xcd, alpha, beta, pruned, with_bias, act, dtype, flush=True)
        assert plan.choice(M, lda, ldc, beta)["shape"] == shape
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
                  pruned_cols=pruned, bias_ptr=dbias.data_ptr() if with_bias else None, activation=act,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, beta, pruned, with_bias, act) in (
                    (1.0, 0.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                    (0.5, 0.0, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                    (1.0, 0.0, tw.PRUNED_ZERO, True, tw.ACT_GELU),
                    (2.0, 0.75, tw.PRUNED_ZERO, False, tw.ACT_NONE)):
                want = launch(plan, tw.SHAPE_128x64, -1, 0, alpha, beta, pruned, with_bias, act)
                for piece, xcd in ((-1, 0), (-1, 1), (32, 0), (32, 1)):
                    got = launch(plan, tw.SHAPE_256x64, piece, xcd, alpha, beta, pruned, with_bias, act)
                    assert np.array_equal(got, want), (piece, xcd, alpha, beta, pruned, with_bias, act)
                assert (want[:, M:] == SENTINEL).all()
                if not with_bias and act == tw.ACT_NONE:
                    Cf = oracle.bits_to_f32(want[:, :M], dtype).reshape(N, M).T
                    ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
                    assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
    finally:
        for opt in (tw.OPT_SHAPE, tw.OPT_PIECE, tw.OPT_XCD_QUEUES):
            tw.set_option(opt, -1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M", [1, 31, 64, 100, 129, 200])
def test_skinny_kernel(tw, oracle, dtype, M):
    """The skinny kernel (32 rows of A and half a unit per workgroup, the kept rows split over its
    waves, the partial sums added in wave order) is what few rows of A get by default.  Tiles from
    no kept row over one step to 23 steps (three rounds of pairs, the last one odd), 7 to 128
    kept columns, ragged M, alpha / beta, bias + activation, filled pruned columns: within half
    the tolerance of the streaming 256 x 128 kernel (the sum over k runs in four slices), bit for
    bit what it gives where nothing is summed (pruned columns, tiles without kept rows), nothing
    written outside, and the same bits on a second launch."""
    rng = np.random.default_rng(555 + M)
    K, N, G = 1500, 768, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = []
    for t, (kt, nt) in enumerate(((1460, 128), (64, 100), (0, 128), (333, 65), (700, 7), (1, 33))):
        tiles.append(dict(col0=t * G, width=G,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(G, size=nt, replace=False)).astype(np.int32)))
    keep = kept_columns(tiles, N)
    import torch
    dbias = torch.from_numpy(bias).cuda()
    lda = ldc = round_up(M, 8) + 8
    At = np.zeros((K, lda), np.uint16)
    At[:, :M] = oracle.cast_bits(A, dtype).reshape(M, K).T
    dA = to_device_bits(At, At.shape)

    def launch(plan, shape, alpha, beta, pruned, with_bias, act):
        Cb = np.full((N, ldc), SENTINEL, np.uint16)
        Cb[:, :M] = oracle.cast_bits(C0, dtype).reshape(M, N).T
        dC = to_device_bits(Cb, Cb.shape)
        tw.set_option(tw.OPT_SHAPE, shape)
        print("skinny test: shape", shape, M, alpha, beta, pruned, with_bias, act, dtype, flush=True)
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta,
                  pruned_cols=pruned, bias_ptr=dbias.data_ptr() if with_bias else None, activation=act,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return from_device_bits(dC)

    no_sum = np.ones(N, bool)                   # columns whose value does not come from a sum over k
    for t in tiles:
        if len(t["kept_k"]):
            no_sum[t["col0"] + t["kept_n"]] = False
    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for (alpha, beta, pruned, with_bias, act) in (
                    (1.0, 0.0, tw.PRUNED_UNTOUCHED, False, tw.ACT_NONE),
                    (0.5, 0.0, tw.PRUNED_ZERO, True, tw.ACT_RELU),
                    (1.0, 0.0, tw.PRUNED_ZERO, True, tw.ACT_TANH),
                    (2.0, 0.75, tw.PRUNED_ZERO, False, tw.ACT_NONE),
                    (1.0, -0.5, tw.PRUNED_UNTOUCHED, True, tw.ACT_GELU)):
                want = launch(plan, tw.SHAPE_256x128, alpha, beta, pruned, with_bias, act)
                got = launch(plan, -1, alpha, beta, pruned, with_bias, act)     # the default: skinny
                forced = launch(plan, tw.SHAPE_SKINNY, alpha, beta, pruned, with_bias, act)
                assert np.array_equal(got, forced)
                assert np.array_equal(got[:, M:], want[:, M:])                  # padding untouched
                if act != tw.ACT_GELU:
                    assert np.array_equal(got[no_sum], want[no_sum])
                a = oracle.bits_to_f32(got[:, :M], dtype)
                b = oracle.bits_to_f32(want[:, :M], dtype)
                assert oracle.rel_error(a, b) <= 0.5 * TOL[dtype], (alpha, beta, pruned, with_bias, act)
                if not with_bias and act == tw.ACT_NONE:
                    Cf = a.reshape(N, M).T
                    ref = reference(oracle, A, B, tiles, dtype, alpha, beta, C0)
                    assert oracle.rel_error(Cf[:, keep], ref[:, keep]) <= TOL[dtype]
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


def test_skinny_kernel_many_units(tw, oracle):
    """More units than travel in the kernel arguments (40 tiles of 64 and 128 columns): the skinny
    kernel reads its unit from the plan's table in memory.  Against the oracle, the streaming
    kernel and itself."""
    rng = np.random.default_rng(909)
    M, K = 96, 700
    widths = [128, 64] * 20
    N = sum(widths)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles, c0 = [], 0
    for t, w in enumerate(widths):
        kt = int(rng.integers(0, 400))
        nt = int(rng.integers(1, w + 1))
        tiles.append(dict(col0=c0, width=w,
                          kept_k=np.sort(rng.choice(K, size=kt, replace=False)).astype(np.int32),
                          kept_n=np.sort(rng.choice(w, size=nt, replace=False)).astype(np.int32)))
        c0 += w
    keep = kept_columns(tiles, N)
    ref = reference(oracle, A, B, tiles, "f16")
    try:
        with tw.Plan.create(K, N, "f16", tiles, B) as plan:
            assert plan.info()["n_tiles"] > 32
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_SKINNY)
            print("skinny, many units: launch", flush=True)
            C1, bits1 = run_gemm(tw, oracle, plan, A, "f16", N, pruned=1)
            C2, bits2 = run_gemm(tw, oracle, plan, A, "f16", N, pruned=1)
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_128x64)
            tw.set_option(tw.OPT_PIECE, 64)
            C3, _ = run_gemm(tw, oracle, plan, A, "f16", N, pruned=1)
            assert np.array_equal(bits1, bits2)
            assert oracle.rel_error(C1[:, keep], ref[:, keep]) <= TOL["f16"]
            assert oracle.rel_error(C1, C3) <= 0.5 * TOL["f16"]
            assert (C1[:, ~keep] == 0).all()
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
        tw.set_option(tw.OPT_PIECE, -1)


@pytest.mark.parametrize("M, K, n_units, width, k_max, dtype", [
    (1, 720, 1, 128, 700, "f16"),       # one row: 31 of the 32 repeat it
    (31, 65, 3, 128, 65, "bf16"),       # a step of one kept row behind a whole one
    (33, 129, 8, 64, 129, "f16"),       # one half per unit, four waves, one row in the last row block
    (500, 720, 5, 128, 256, "bf16"),    # four waves with a step each
    (200, 3001, 9, 128, 2000, "f16"),   # eight waves with several steps, K too long for a panel of A
])
def test_skinny_row_major_gives_the_k_major_bits(tw, oracle, M, K, n_units, width, k_max, dtype):
    """The skinny kernel on row-major A and C: bit for bit its result on K-major copies, with NaN in the
    rows no tile keeps, beta, bias and filled pruned columns; nothing written outside M x N."""
    import torch
    rng = np.random.default_rng([M, K, n_units])
    N = n_units * width
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    tiles = [dict(col0=t * width, width=width,
                  kept_k=np.sort(rng.choice(K, size=k_max if t == 0 else int(rng.integers(0, k_max)),
                                            replace=False)).astype(np.int32),
                  kept_n=np.sort(rng.choice(width, size=int(rng.integers(1, width + 1)),
                                            replace=False)).astype(np.int32)) for t in range(n_units)]
    A[:, np.setdiff1d(np.arange(K), np.concatenate([t["kept_k"] for t in tiles]))] = np.nan
    Ab, Cb = oracle.cast_bits(A, dtype).reshape(M, K), oracle.cast_bits(C0, dtype).reshape(M, N)
    lda, ldc, ldm = round_up(K, 8) + 8, round_up(N, 8) + 8, round_up(M, 8)
    Ar, Cr = np.zeros((M, lda), np.uint16), np.full((M, ldc), SENTINEL, np.uint16)
    Ak, Ck = np.zeros((K, ldm), np.uint16), np.full((N, ldm), SENTINEL, np.uint16)
    Ar[:, :K], Cr[:, :N], Ak[:, :M], Ck[:, :M] = Ab, Cb, Ab.T, Cb.T
    bias = torch.randn(N, device="cuda")
    try:
        tw.set_option(tw.OPT_SHAPE, tw.SHAPE_SKINNY)
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for kw in (dict(pruned_cols=tw.PRUNED_UNTOUCHED),
                       dict(pruned_cols=tw.PRUNED_ZERO, alpha=0.5, beta=2.0, bias_ptr=bias.data_ptr(),
                            activation=tw.ACT_GELU)):
                print("skinny row-major", M, K, n_units, flush=True)
                dA, dC, dAk, dCk = (to_device_bits(x, x.shape) for x in (Ar, Cr, Ak, Ck))
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, a_layout=tw.ROWMAJOR,
                          c_layout=tw.ROWMAJOR, **kw)
                plan.gemm(dAk.data_ptr(), dCk.data_ptr(), M, lda=ldm, ldc=ldm, **kw)
                torch.cuda.synchronize()
                have, want = from_device_bits(dC), from_device_bits(dCk)
                assert np.array_equal(have[:, :N], np.ascontiguousarray(want[:, :M].T))
                assert np.all(have[:, N:] == SENTINEL)
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


@pytest.mark.parametrize("row_major", [False, True])
@pytest.mark.parametrize("n_units, width, k_max, rows, dtype", [
    (11, 128, 700, 33, "f16"), (8, 128, 250, 32, "bf16"), (3, 96, 1000, 50, "f16"), (16, 64, 130, 64, "bf16"), (5, 40, 600, 7, "f16")])
def test_skinny_pieces_give_the_same_bits(tw, oracle, n_units, width, k_max, rows, dtype, row_major):
    """Few rows run in pieces of 32 columns, many in pieces of 64: the first rows of a launch with enough of them to
    fill the chip more than twice are bit for bit those of a launch with these rows alone."""
    import torch
    rng = np.random.default_rng([n_units, width, k_max])
    K, N = 1040, n_units * width
    M = 32 * (2 * 256 * 2 // (n_units * 2) + 1)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = [dict(col0=t * width, width=width,
                  kept_k=np.sort(rng.choice(K, size=k_max if t == 0 else int(rng.integers(0, k_max)),
                                            replace=False)).astype(np.int32),
                  kept_n=np.sort(rng.choice(width, size=int(rng.integers(1, width + 1)),
                                            replace=False)).astype(np.int32)) for t in range(n_units)]
    layout = tw.ROWMAJOR if row_major else tw.KMAJOR
    Ab = oracle.cast_bits(rng.standard_normal((M, K)).astype(np.float32), dtype).reshape(M, K)
    bias = torch.randn(N, device="cuda")
    outs = []
    try:
        tw.set_option(tw.OPT_SHAPE, tw.SHAPE_SKINNY)
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            for m in (rows, M):
                ld = round_up(m, 8)
                host = Ab[:m] if row_major else np.zeros((K, ld), np.uint16)
                if not row_major:
                    host[:, :m] = Ab[:m].T
                dA = to_device_bits(host, host.shape)
                dC = torch.zeros((m, N) if row_major else (N, ld), dtype=torch.int16, device="cuda")
                print("skinny pieces", n_units, width, k_max, m, dtype, row_major, flush=True)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), m, lda=host.shape[1], ldc=dC.shape[1], a_layout=layout, c_layout=layout,
                          pruned_cols=tw.PRUNED_ZERO, bias_ptr=bias.data_ptr(), activation=tw.ACT_RELU)
                torch.cuda.synchronize()
                outs.append(from_device_bits(dC)[:rows] if row_major else from_device_bits(dC)[:, :rows])
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n_units", [1, 2, 3, 4, 5, 7, 8, 11])
@pytest.mark.parametrize("M", [1, 33, 500])
@pytest.mark.parametrize("k_max, width", [(256, 128), (700, 128), (256, 64)])
def test_skinny_work_split(tw, oracle, n_units, M, k_max, width):
    """How the skinny kernel hands its work out: units in groups of eight, the ones left over on a
    set of dies each (row blocks in turn, so workgroups of a row block past the last leave at once),
    one half or two per unit, four waves (256 kept rows at most) or eight.  Against the oracle, with
    nothing written outside."""
    rng = np.random.default_rng([n_units, M, k_max, width])
    K, N = 720, n_units * width
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = [dict(col0=t * width, width=width,
                  kept_k=np.sort(rng.choice(K, size=k_max if t == 0 else int(rng.integers(0, k_max)),
                                            replace=False)).astype(np.int32),
                  kept_n=np.sort(rng.choice(width, size=int(rng.integers(1, width + 1)),
                                            replace=False)).astype(np.int32)) for t in range(n_units)]
    keep = kept_columns(tiles, N)
    try:
        with tw.Plan.create(K, N, "f16", tiles, B) as plan:
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_SKINNY)
            print("skinny split", n_units, M, k_max, width, flush=True)
            C, bits = run_gemm(tw, oracle, plan, A, "f16", N, pad=8)
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)
    ref = reference(oracle, A, B, tiles, "f16")
    assert oracle.rel_error(C[:, keep], ref[:, keep]) <= TOL["f16"]
    assert np.all(bits[~keep, :] == SENTINEL) and np.all(bits[:, M:] == SENTINEL)


def test_operand_beyond_four_gib(tw, oracle):
    """A of 4.4 GiB: byte offsets into A no longer fit 32 bits, the launch falls back to the
    kernel with 64-bit addressing.  Checked on sampled rows (a row of C depends on the same row
    of A only) at both ends of M."""
    import torch
    K, N, G = 2304, 128, 128
    M = 1024 * 1000                        # K * M * 2 bytes = 4.4 GiB
    rng = np.random.default_rng(99)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.25, n_keep=0.9)
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    dA = torch.empty((K, M), dtype=torch.float16, device="cuda")
    for k0 in range(0, K, 256):            # filled in slabs: no 2x temporary
        dA[k0:k0 + 256].normal_(generator=g)
    dC = torch.full((N, M), 7.0, dtype=torch.float16, device="cuda")
    print("4 GiB operand: launch", flush=True)
    with tw.Plan.create(K, N, "f16", tiles, B) as plan:
        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    rows = np.concatenate([np.arange(0, 40), rng.integers(0, M, 60), np.arange(M - 40, M)])
    idx = torch.from_numpy(rows).cuda()
    A_rows = dA[:, idx].float().cpu().numpy().T          # [rows, K], exact fp16 values
    C_rows = dC[:, idx].float().cpu().numpy().T
    ref = oracle.tw_gemm_reference(A_rows, oracle.quantize(B, "f16"), tiles)
    keep = kept_columns(tiles, N)
    assert oracle.rel_error(C_rows[:, keep], ref[:, keep]) <= 1e-2
    assert np.all(C_rows[:, ~keep] == 7.0)               # pruned columns untouched


def test_concurrent_host_threads_and_streams(tw, oracle):
    """One immutable plan, four host threads, each launching on its own stream into its own C:
    every thread gets the single-stream result bit for bit."""
    import threading
    import torch
    rng = np.random.default_rng(111)
    M, K, N, G = 1024, 384, 512, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.9)
    At = np.ascontiguousarray(oracle.cast_bits(A, "f16").reshape(M, K).T)
    dA = to_device_bits(At, At.shape)
    with tw.Plan.create(K, N, "f16", tiles, B) as plan:
        want = torch.zeros((N, M), dtype=torch.int16, device="cuda")
        plan.gemm(dA.data_ptr(), want.data_ptr(), M, pruned_cols=tw.PRUNED_ZERO,
                  stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs = [torch.full((N, M), 0x1234, dtype=torch.int16, device="cuda") for _ in range(4)]
        streams = [torch.cuda.Stream() for _ in range(4)]
        errors = []

        def work(i):
            try:
                for _ in range(60):
                    plan.gemm(dA.data_ptr(), outs[i].data_ptr(), M, pruned_cols=tw.PRUNED_ZERO,
                              stream=streams[i].cuda_stream)
                streams[i].synchronize()
            except Exception as e:           # surfaced by the main thread
                errors.append(e)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for o in outs:
            assert torch.equal(o, want)


@pytest.mark.parametrize("M,K,N,kept,skinny", [
    # workgroups of the kernel for few rows to a compute unit of the fullest of eight dies (of 32 units each): w
    (1024, 768, 2048, 192, True),       # w 4, four-wave form, a panel of A fits LDS
    (1280, 768, 2048, 192, False),      # w 5
    (3072, 768, 768, 192, False),       # w 6: six units leave two dies without work
    (4096, 384, 512, 250, False),       # w 4, more than 2048 rows, tiles not short
    (512, 768, 3072, 448, True),        # w 3, eight-wave form
    (3072, 512, 512, 300, False),       # w 3, more than 1536 rows
    (2048, 512, 1024, 300, False),      # w 4
    (768, 2048, 2048, 1024, True),      # w 3, a 32-row panel fits
    (768, 1536, 3072, 384, False),      # w 4.5
    (2560, 2048, 768, 500, True),       # w 5, streaming items of 64 columns
    (2560, 4608, 1024, 460, False),     # w 5, streaming items of 256 x 128
    (1536, 1536, 2048, 150, True),      # w 6, four-wave form
    (3072, 3072, 768, 310, False),      # w 6
])
def test_kernel_for_few_rows_is_taken_where_it_is_ahead(tw, M, K, N, kept, skinny):
    """Both sides of the lines of the launch's rule, at problems whose two kernels were timed."""
    tiles = [dict(col0=c, width=128, kept_k=np.arange(kept, dtype=np.int32), kept_n=np.arange(128, dtype=np.int32))
             for c in range(0, N, 128)]
    with tw.Plan.create(K, N, "f16", tiles, np.zeros((K, N), np.float32)) as plan:
        assert (plan.choice(M, round_up(M, 64), round_up(M, 64))["shape"] == tw.SHAPE_SKINNY) == skinny


@pytest.mark.parametrize("M,K,N,G,k_keep,n_keep,dtype", [
    (1100, 2203, 1530, 128, 0.25, 1.0, "f16"),    # ragged M, K and N; whole octets of columns
    (1100, 2203, 1530, 128, 0.25, 0.8, "bf16"),   # element-wise stores
    (1600, 2136, 1000, 64, 0.3, 1.0, "f16"),      # units of at most 64 columns: a wave each
    (1300, 3000, 1290, 128, 0.01, 0.9, "f16"),    # groups of 16 kept rows over many chunks: cut
    (3080, 2400, 520, 128, 0.6, 0.9, "bf16"),     # a last group of units that is not full
    (4096, 1024, 1024, 128, 0.25, 1.0, "f16"),    # where a panel of A would fit
])
def test_row_major_streaming(tw, oracle, M, K, N, G, k_keep, n_keep, dtype):
    """Row-major A and C through the row-major streaming kernel (forced: some of these calls take another by themselves): alpha, bias
    and ReLU, pruned columns left alone, then beta and pruned columns filled; tiles without kept rows; padding and
    the workspace untouched (nothing is staged).  Sampled rows against the oracle."""
    import torch
    rng = np.random.default_rng(M + K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=k_keep, n_keep=n_keep, empty_every=5)
    keep = kept_columns(tiles, N)
    lda, ldc = round_up(K, 8) + 8, round_up(N, 8) + 8
    Ah, Ch = np.full((M, lda), 0x7e00 if dtype == "f16" else 0x7fc0, np.uint16), np.full((M, ldc), SENTINEL, np.uint16)
    Ah[:, :K] = oracle.cast_bits(A, dtype).reshape(M, K)       # NaN in the padding of the rows of A
    Ch[:, :N] = oracle.cast_bits(C0, dtype).reshape(M, N)
    dA, d_bias = to_device_bits(Ah, Ah.shape), torch.from_numpy(bias).cuda()
    rows = np.unique(np.concatenate([np.arange(5), np.arange(M - 70, M), rng.choice(M, 40)]))
    try:
        tw.set_option(tw.OPT_SHAPE, tw.SHAPE_RM)
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            nbytes = max(plan.staged_workspace(M, tw.ROWMAJOR, tw.ROWMAJOR), 16)
            ws = torch.full((nbytes // 2,), 0x7bcd, dtype=torch.int16, device="cuda")
            for alpha, beta, pruned in ((0.75, 0.0, tw.PRUNED_UNTOUCHED), (1.0, 0.5, tw.PRUNED_ZERO)):
                dC = to_device_bits(Ch, Ch.shape)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta, a_layout=tw.ROWMAJOR,
                          c_layout=tw.ROWMAJOR, pruned_cols=pruned, bias_ptr=d_bias.data_ptr(), activation=tw.ACT_RELU,
                          workspace_ptr=ws.data_ptr(), workspace_bytes=nbytes)
                torch.cuda.synchronize()
                assert torch.all(ws == 0x7bcd)
                out = from_device_bits(dC)
                assert np.all(out[:, N:] == SENTINEL)
                pre = alpha * reference(oracle, A[rows], B, tiles, dtype)
                want = np.maximum(pre + beta * oracle.quantize(C0[rows], dtype) + bias, 0.0)
                got = oracle.bits_to_f32(np.ascontiguousarray(out[rows, :N]), dtype).reshape(rows.size, N)
                assert oracle.rel_error(got[:, keep], want[:, keep]) <= TOL[dtype]
                if pruned == tw.PRUNED_UNTOUCHED:
                    assert np.array_equal(out[:, :N][:, ~keep], Ch[:, :N][:, ~keep])
                elif not np.all(keep):
                    assert oracle.rel_error(got[:, ~keep], want[:, ~keep]) <= TOL[dtype]
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


def test_row_major_streaming_nonfinite(tw, oracle):
    """Inf and NaN in columns of A that a tile prunes do not reach it, and an infinite weight in a group of kept rows that
    is cut gives what it gives uncut: the row-major streaming kernel and the K-major one agree on where the result is finite."""
    import torch
    rng = np.random.default_rng(5)
    M, K, N, G = 1100, 2500, 1536, 128
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=0.02, n_keep=1.0)
    free = np.setdiff1d(np.arange(K), np.concatenate([t["kept_k"] for t in tiles[:6]]))
    A[:, free[::3]], A[:, free[1::3]] = np.inf, np.nan         # (kept by other tiles: those become non-finite)
    A[A == 0] = 1.0
    for t in tiles[:3]:
        B[t["kept_k"][7], t["col0"] + 11] = 1e9                # infinite in f16
    Ak = np.zeros((K, round_up(M, 8)), np.uint16)
    Ab = oracle.cast_bits(A, "f16").reshape(M, K)
    Ak[:, :M] = Ab.T
    Ar = np.zeros((M, round_up(K, 8)), np.uint16)
    Ar[:, :K] = Ab
    dAk, dAr = to_device_bits(Ak, Ak.shape), to_device_bits(Ar, Ar.shape)
    dCk, dCr = (torch.zeros(s, dtype=torch.int16, device="cuda") for s in ((N, Ak.shape[1]), (M, N)))
    with tw.Plan.create(K, N, "f16", tiles, B) as plan:
        try:
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_RM)
            assert plan.kernel_name(M, Ar.shape[1], N, tw.ROWMAJOR, tw.ROWMAJOR) == "tw_gemm_rm_kernel"
            plan.gemm(dAr.data_ptr(), dCr.data_ptr(), M, lda=Ar.shape[1], ldc=N, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR)
        finally:
            tw.set_option(tw.OPT_SHAPE, -1)
        plan.gemm(dAk.data_ptr(), dCk.data_ptr(), M, lda=Ak.shape[1], ldc=Ak.shape[1])
        torch.cuda.synchronize()
    r, k = dCr.view(torch.float16), dCk.view(torch.float16)[:, :M].T
    assert torch.equal(torch.isnan(r), torch.isnan(k)) and torch.equal(torch.isinf(r), torch.isinf(k))
    assert bool(torch.isfinite(r[:, :6 * G]).any()) and bool(torch.isinf(r[:, 11]).all())
    fin = torch.isfinite(r)
    assert float((r[fin].float() - k[fin].float()).abs().max()) <= 2e-3 * float(k[fin].float().abs().max())


@pytest.mark.parametrize("M,K,N,G,k_keep,n_keep,act,dtype", [
    (300, 2203, 1530, 128, 0.25, 0.9, "gelu", "f16"),    # ragged; 12 units, read from the arguments
    (130, 2500, 4400, 128, 0.2, 1.0, "tanh", "bf16"),    # 35 units: read from memory
    (200, 2300, 2200, 64, 0.02, 0.9, "gelu", "bf16"),    # units of at most 64 columns, a wave each; groups cut
    (70, 3000, 330, 64, 0.01, 1.0, "relu", "f16"),
    (64, 100, 128, 128, 0.5, 1.0, "none", "bf16"),       # one chunk of K, one unit: waves and loading waves without work
    (65, 260, 200, 32, 0.9, 0.8, "tanh", "f16"),
    (4096, 1024, 1024, 128, 0.25, 1.0, "gelu", "f16"),
])
def test_row_major_streaming_forced(tw, oracle, M, K, N, G, k_keep, n_keep, act, dtype):
    """The row-major streaming kernel wherever it can run, forced and named: every activation, bias, alpha, C read and not read,
    pruned columns filled and left alone, tiles without kept rows.  Sampled rows against the oracle."""
    import torch
    rng = np.random.default_rng(M + K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    tiles = random_tiles(rng, K, N, G, k_keep=k_keep, n_keep=n_keep, empty_every=5)
    keep = kept_columns(tiles, N)
    lda, ldc = round_up(K, 8) + 8, round_up(N, 8) + 8
    Ah, Ch = np.full((M, lda), 0x7e00 if dtype == "f16" else 0x7fc0, np.uint16), np.full((M, ldc), SENTINEL, np.uint16)
    Ah[:, :K] = oracle.cast_bits(A, dtype).reshape(M, K)
    Ch[:, :N] = oracle.cast_bits(C0, dtype).reshape(M, N)
    dA, d_bias = to_device_bits(Ah, Ah.shape), torch.from_numpy(bias).cuda()
    code = {"none": tw.ACT_NONE, "relu": tw.ACT_RELU, "gelu": tw.ACT_GELU, "tanh": tw.ACT_TANH}[act]
    rows = np.unique(np.concatenate([np.arange(min(M, 40)), np.arange(max(0, M - 70), M), rng.choice(M, 20)]))
    row = dict(a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR)
    try:
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            tw.set_option(tw.OPT_SHAPE, tw.SHAPE_RM)
            for alpha, beta, pruned in ((0.75, 0.0, tw.PRUNED_UNTOUCHED), (1.0, 0.5, tw.PRUNED_ZERO)):
                assert plan.kernel_name(M, lda, ldc, beta=beta, activation=code, **row) == "tw_gemm_rm_kernel"
                dC = to_device_bits(Ch, Ch.shape)
                print("row-major streaming, forced:", M, K, N, G, beta, act, dtype, flush=True)
                plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=lda, ldc=ldc, alpha=alpha, beta=beta, pruned_cols=pruned,
                          bias_ptr=d_bias.data_ptr(), activation=code, **row)
                torch.cuda.synchronize()
                out = from_device_bits(dC)
                assert np.all(out[:, N:] == SENTINEL)
                pre = alpha * reference(oracle, A[rows], B, tiles, dtype).astype(np.float64)
                want = oracle.ACTIVATIONS[act](pre + beta * oracle.quantize(C0[rows], dtype) + bias)
                got = oracle.bits_to_f32(np.ascontiguousarray(out[rows, :N]), dtype).reshape(rows.size, N)
                assert oracle.rel_error(got[:, keep], want[:, keep]) <= TOL[dtype]
                if pruned == tw.PRUNED_UNTOUCHED:
                    assert np.array_equal(out[:, :N][:, ~keep], Ch[:, :N][:, ~keep])
                elif not np.all(keep):
                    assert oracle.rel_error(got[:, ~keep], want[:, ~keep]) <= TOL[dtype]
    finally:
        tw.set_option(tw.OPT_SHAPE, -1)


ROUTES = [
    # M, K, N, G, kept rows, beta, workspace -> kernel.  The ways a row-major call takes at both sides of their lines
    (4096, 3072, 768, 128, 768, 0.0, "tw_gemm_rm_kernel"),                 # BERT-base's second layer
    (4096, 1024, 1024, 128, 256, 0.0, "tw_gemm_as_kernel 64 rows row-major"),
    (4096, 2048, 1024, 128, 512, 0.0, "tw_gemm_as_kernel 32 rows row-major"),
    (1863, 3544, 856, 128, 7, 0.0, "tw_gemm_skinny_kernel row-major"),     # (hardly any row kept, short walks)
    (2048, 3072, 768, 128, 768, 0.0, "tw_gemm_skinny_kernel row-major"),
    (2600, 3072, 768, 128, 768, 0.0, "tw_gemm_rm_kernel"),
    (128, 3072, 768, 128, 768, 0.0, "tw_gemm_skinny_kernel row-major"),
    (6123, 3536, 5248, 128, 18, 0.0, "tw_gemm_generic_kernel"),            # staged where there is a workspace
    (2968, 3352, 2608, 64, 1676, 0.0, "tw_gemm_rm_kernel"),                # (the same: without one)
    (6000, 400, 2000, 128, 100, 0.5, "tw_gemm_rm_kernel"),
    (6000, 3300, 2000, 128, 40, 0.5, "tw_gemm_generic_kernel"),
]


@pytest.mark.parametrize("M,K,N,G,kept,beta,kernel", ROUTES)
def test_which_kernel_takes_row_major_operands(tw, M, K, N, G, kept, beta, kernel):
    tiles = [dict(col0=c, width=min(G, N - c), kept_k=np.arange(kept, dtype=np.int32), kept_n=np.arange(min(G, N - c), dtype=np.int32))
             for c in range(0, N, G)]
    with tw.Plan.create(K, N, "f16", tiles, np.zeros((K, N), np.float32)) as plan:
        assert plan.kernel_name(M, K, N, tw.ROWMAJOR, tw.ROWMAJOR, beta=beta) == kernel


@pytest.mark.parametrize("staged,M", [(False, 8), (True, 8), (False, 8200)])
def test_row_major_operands_with_more_units_than_a_grid_has_rows(tw, staged, M):
    """262208 tiles of one column: more groups of units than the second dimension of a grid has.  Row-major calls of such a
    plan run on the kernels that number their workgroups in one dimension, with a workspace and without; 8200 rows are more
    work items than one launch takes."""
    import torch
    K, N = 16, 262208
    gen = torch.Generator("cuda").manual_seed(3)
    A = torch.randn((M, K), generator=gen, device="cuda").half()
    B = torch.randn((K, N), generator=gen, device="cuda")
    C0 = torch.randn((M, N), generator=gen, device="cuda").half()
    kept = torch.arange(N, device="cuda") % K                # the one kept row of every tile
    mask = torch.zeros((K, N), dtype=torch.uint8, device="cuda")
    mask[kept, torch.arange(N, device="cuda")] = 1
    rows = torch.unique(torch.tensor([0, 1, 2, 3, 4, 5, 6, 7, 127, 128, 8063, 8064, 8191, 8192, 8199], device="cuda").clamp(max=M - 1))
    want = A[rows].double()[:, kept] * B.half().double()[kept, torch.arange(N, device="cuda")] + 0.5 * C0[rows].double()
    s = torch.cuda.current_stream().cuda_stream
    with tw.Plan.from_device_mask(K, N, mask.data_ptr(), [(c, 1) for c in range(N)], "f16", B.data_ptr(), stream=s) as plan:
        nbytes = plan.staged_workspace(M, tw.ROWMAJOR, tw.ROWMAJOR) if staged else 0
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if staged else None
        C = C0.clone()
        plan.gemm(A.data_ptr(), C.data_ptr(), M, lda=K, ldc=N, beta=0.5, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR, stream=s,
                  workspace_ptr=ws.data_ptr() if staged else None, workspace_bytes=nbytes)
        torch.cuda.synchronize()
    # one product in fp32, one rounding to f16
    assert bool(((C[rows].double() - want).abs() <= 2.0 ** -11 * want.abs() * 1.01 + 1e-6).all())


@pytest.mark.parametrize("beta", [2.0, 0.0])
def test_row_major_operands_with_more_rows_than_a_grid_takes_threads(tw, beta):
    """2^29 + 70 rows: a workgroup for every 64 of them is beyond 2^32 threads, with C read (no panel of A in LDS then) and not
    read (a panel)."""
    import torch
    M, K, N = (1 << 29) + 70, 8, 8
    B = torch.full((K, N), 0.5, device="cuda")
    mask = torch.zeros((K, N), dtype=torch.uint8, device="cuda")
    mask[2:5] = 1
    s = torch.cuda.current_stream().cuda_stream
    A = torch.ones((M, K), dtype=torch.float16, device="cuda")
    A[-3:] = 2.0
    A[:, 0] = 7.0                                            # (not kept)
    C = torch.ones((M, N), dtype=torch.float16, device="cuda")
    with tw.Plan.from_device_mask(K, N, mask.data_ptr(), [(0, N)], "f16", B.data_ptr(), stream=s) as plan:
        plan.gemm(A.data_ptr(), C.data_ptr(), M, lda=K, ldc=N, beta=beta, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR, stream=s)
        torch.cuda.synchronize()
    assert bool((C[-3:] == 3.0 + beta).all()) and bool((C[:100] == 1.5 + beta).all()) and bool((C[M - 200:-3] == 1.5 + beta).all())
    assert int((C != 1.5 + beta).sum(dtype=torch.int64)) == 3 * N


@pytest.mark.parametrize("shape,G,blocks", [("128x32", 32, 7), ("128x32", 32, 40), ("128x32", 32, 43), ("256x64", 64, 43)])
@pytest.mark.parametrize("pruned", ["untouched", "zero"])
def test_queues_of_the_dies_hand_out_every_item_once(tw, oracle, shape, G, blocks, pruned):
    """Row blocks owned by the dies, items dealt out tile after tile and row block after row block: fewer row blocks
    than dies (nobody owns one), five to a die in a group of two and one of three, the same with three
    left over, each with one to a die's share of a launch and with twelve items and more to a workgroup (the
    256-row items only in fewer workgroups), tiles without kept rows and pruned columns to fill among them.  Every
    launch starts from the same C and adds half of it, so that an item left out, or taken up again after it was
    stored, differs from the oracle; nothing but the products' columns is written."""
    import torch
    rng = np.random.default_rng(5 + blocks)
    K, N = 96, 2688
    rows = int(shape.split("x")[0])
    tiles = random_tiles(rng, K, N, G, k_keep=0.4, n_keep=0.7, empty_every=20)
    B = (rng.standard_normal((K, N)) * 0.1).astype(np.float32)
    M = blocks * rows - 5
    ld = round_up(M, 8)
    A = rng.standard_normal((M, K)).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    want = reference(oracle, A, B, tiles, "f16", beta=0.5, C0=C0).T
    start = np.full((N, ld), SENTINEL, np.uint16)
    start[:, :M] = oracle.cast_bits(C0, "f16").reshape(M, N).T
    At = np.zeros((K, ld), np.uint16)
    At[:, :M] = oracle.cast_bits(A, "f16").reshape(M, K).T
    dA, dstart = to_device_bits(At, At.shape), to_device_bits(start, start.shape)
    keep = kept_columns(tiles, N)
    if pruned == "zero":
        want[~keep] = 0.5 * oracle.quantize(C0, "f16").T[~keep]
    got = []
    try:
        with tw.Plan.create(K, N, "f16", tiles, B) as plan:
            tw.set_option(tw.OPT_SHAPE, getattr(tw, "SHAPE_" + shape))
            tw.set_option(tw.OPT_PIECE, 32)
            for per_cu in (1, 8):
                tw.set_option(tw.OPT_WGS_PER_CU, per_cu)
                for xcd in (0, 1, 2, -1):
                    tw.set_option(tw.OPT_XCD_QUEUES, xcd)
                    print("queues", shape, blocks, pruned, per_cu, xcd, flush=True)
                    for _ in range(2):  # (the second launch finds the counters as the first left them)
                        dC = dstart.clone()
                        plan.gemm(dA.data_ptr(), dC.data_ptr(), M, lda=ld, ldc=ld, beta=0.5,
                                  pruned_cols=tw.PRUNED_ZERO if pruned == "zero" else tw.PRUNED_UNTOUCHED,
                                  stream=torch.cuda.current_stream().cuda_stream)
                        got.append(dC)
    finally:
        for opt in (tw.OPT_SHAPE, tw.OPT_PIECE, tw.OPT_WGS_PER_CU, tw.OPT_XCD_QUEUES):
            tw.set_option(opt, -1)
    first = from_device_bits(got[0])
    written = oracle.bits_to_f32(first[:, :M], "f16").reshape(N, M)
    assert (first[:, M:] == SENTINEL).all()
    if pruned == "untouched":
        assert np.array_equal(first[~keep], start[~keep])
        written, want = written[keep], want[keep]
    # one rounding to 16 bits (2^-11 of the result), and 39 kept rows' products added in 32 bits
    assert (np.abs(written - want) <= 2.0 ** -11 * np.abs(want) + 1e-5).all()
    assert all(torch.equal(got[0], g) for g in got)


def test_choice_names_queues_of_kernels_that_have_them(tw, oracle):
    """choice()'s xcd_queues: only for a kernel that draws its items from queues, and as the options ask."""
    rng = np.random.default_rng(9)
    tiles = random_tiles(rng, 256, 512, 64, k_keep=0.3)
    B = rng.standard_normal((256, 512)).astype(np.float32)
    queued = {tw.SHAPE_WIDE, tw.SHAPE_128x128, tw.SHAPE_512x64, tw.SHAPE_128x64, tw.SHAPE_256x128, tw.SHAPE_128x32, tw.SHAPE_256x64}
    seen = set()
    try:
        with tw.Plan.create(256, 512, "f16", tiles, B) as plan:
            for shape in range(13):
                tw.set_option(tw.OPT_SHAPE, shape)
                for xcd in (-1, 0, 1, 2):
                    tw.set_option(tw.OPT_XCD_QUEUES, xcd)
                    c = plan.choice(4096)
                    seen.add(c["shape"])
                    assert c["xcd_queues"] == (c["shape"] in queued and xcd in (-1, 1)), (shape, xcd, c)
                tw.set_option(tw.OPT_XCD_QUEUES, -1)
                tw.set_option(tw.OPT_BALANCE, 1)
                assert not plan.choice(4096)["xcd_queues"]
                tw.set_option(tw.OPT_BALANCE, -1)
    finally:
        for opt in (tw.OPT_SHAPE, tw.OPT_XCD_QUEUES, tw.OPT_BALANCE):
            tw.set_option(opt, -1)
    assert len(seen & queued) >= 5 and len(seen - queued) >= 3


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 24, 33, 130])
@pytest.mark.parametrize("K,k_keep", [(600, 0.3), (900, 0.4)])     # four waves, and eight
def test_row_major_blocks_of_fewer_rows(tw, oracle, K, k_keep, M, dtype):
    """The kernel for few rows takes 8, 16 or 32 rows of a row-major A a workgroup, by how many workgroups that makes: last blocks of one
    row, whole ones, and a plan so wide that 32 remain.  A row that is no number stays in its own row of C, and no row behind
    the last is written.  The same launch on a single row gives the same bits for every row (the sums do not depend on the block)."""
    import torch
    for N in (96, 2048):
        rng = np.random.default_rng(K + M + N)
        tiles = random_tiles(rng, K, N, 128, k_keep=k_keep, n_keep=0.9)
        B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
        A = rng.standard_normal((M, K)).astype(np.float32)
        lda, ldc, rows = round_up(K, 8), round_up(N, 8), M + 40
        Ab = np.zeros((M, lda), np.uint16)
        Ab[:, :K] = oracle.cast_bits(A, dtype).reshape(M, K)
        if M > 4:
            Ab[3, :K] = 0x7FFF  # NaN in either type
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:
            assert "skinny" in plan.kernel_name(M, lda=lda, ldc=ldc, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR)
            dA = to_device_bits(Ab, Ab.shape)

            def run(first, m):
                dC = to_device_bits(np.full((rows, ldc), 0x1234, np.uint16), (rows, ldc))
                plan.gemm(dA.data_ptr() + first * lda * 2, dC.data_ptr(), m, lda=lda, ldc=ldc, a_layout=tw.ROWMAJOR, c_layout=tw.ROWMAJOR,
                          pruned_cols=tw.PRUNED_ZERO, stream=torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                got = from_device_bits(dC)
                assert (got[m:] == 0x1234).all()
                return got[:m, :N]
            got = run(0, M)
            keep = kept_columns(tiles, N)
            for m in sorted({0, M // 2, M - 1}):
                if M > 4 and m == 3:
                    continue
                assert np.array_equal(got[m], run(m, 1)[0]), (N, m)
            C = oracle.bits_to_f32(got, dtype).reshape(M, N)
            good = [m for m in range(M) if not (M > 4 and m == 3)]
            ref = oracle.quantize(A, dtype).astype(np.float64) @ (oracle.quantize(B, dtype) * oracle.plan_mask(K, N, tiles)).astype(np.float64)
            assert oracle.rel_error(C[good], ref[good]) <= {"f16": 1e-2, "bf16": 2e-2}[dtype]
            if M > 4:
                assert np.isnan(C[3, keep]).all() and (C[3, ~keep] == 0).all()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 24, 33, 130])
@pytest.mark.parametrize("K,k_keep", [(600, 0.3), (900, 0.4)])     # four waves, and eight
def test_k_major_blocks_of_fewer_rows(tw, oracle, K, k_keep, M, dtype):
    """The same of a K-major A, whose rows of a block are one, two or four pieces of a kept row: neither a column that is no number, nor
    the padding behind the last, nor a row that no tile keeps reaches another's result, nothing behind the last column of C is written,
    and a column alone gives the same bits as among the others."""
    import torch
    for N in (96, 1024, 4096):
        rng = np.random.default_rng(K + M + N)
        tiles = random_tiles(rng, K, N, 128, k_keep=k_keep, n_keep=0.9)
        B = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
        A = rng.standard_normal((M, K)).astype(np.float32)
        bits = oracle.cast_bits(A, dtype).reshape(M, K)
        mask = oracle.plan_mask(K, N, tiles)
        bits[:, ~mask.astype(bool).any(1)] = 0x7FFF  # NaN in either type
        if M > 4:
            bits[3] = 0x7FFF
        with tw.Plan.create(K, N, dtype, tiles, B) as plan:

            def run(rows):
                m, ld = rows.shape[0], round_up(rows.shape[0], 8) + 8
                assert "skinny" in plan.kernel_name(m, lda=ld, ldc=ld)
                At = np.full((K, ld), 0x7FFF, np.uint16)
                At[:, :m] = rows.T
                dA, dC = to_device_bits(At, (K, ld)), to_device_bits(np.full((N, ld), 0x1234, np.uint16), (N, ld))
                plan.gemm(dA.data_ptr(), dC.data_ptr(), m, lda=ld, ldc=ld, pruned_cols=tw.PRUNED_ZERO, stream=torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                got = from_device_bits(dC)
                assert (got[:, m:] == 0x1234).all()
                return np.ascontiguousarray(got[:, :m].T)
            got = run(bits)
            keep = kept_columns(tiles, N)
            good = [m for m in range(M) if not (M > 4 and m == 3)]
            for m in sorted({0, M // 2, M - 1} & set(good)):
                assert np.array_equal(got[m], run(bits[m:m + 1])[0]), (N, m)
            C = oracle.bits_to_f32(got, dtype).reshape(M, N)
            ref = oracle.quantize(A, dtype).astype(np.float64) @ (oracle.quantize(B, dtype) * mask).astype(np.float64)
            assert oracle.rel_error(C[good], ref[good]) <= {"f16": 1e-2, "bf16": 2e-2}[dtype]
            if M > 4:
                assert np.isnan(C[3, keep]).all() and (C[3, ~keep] == 0).all()
