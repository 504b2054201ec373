"""The work that users of this engine have it do, as cases that can be timed.

The engine runs pruned networks and prunes them.  Running: masked dense layers and feed-forward
pairs (K-major operands as the engine's own layout has them, or row-major ones as the Python
operator ``x @ (kernel * mask) + bias`` has them), convolutions as im2col products, LSTM cells by
the step and by the sequence.  Pruning: masks from importance scores, and plans from those masks.
Shapes are those of the repository's configurations (BERT-base and BERT-large feed-forward layers,
VGG16 convolutions, the NMT recurrence, the load-imbalance stress, the reference's own driver
command line), at full batches and at the small and odd ones a service sees.

A case's ``kind`` says what it runs:

  dense   one masked layer, C = act(A (B . mask) + bias)
  ffn     two masked layers with GELU between them, K -> N -> K
  lstm    ``steps`` time steps of a cell with ``hidden`` units and as many inputs
  prune   masks for a network of ``layers`` from scores: how = 1d, 2d or 1dmix
  replan  what a pruning round ends with: new 2d masks, a plan for every layer from them, and
          the first product of each plan

The number of kept rows of every column tile belongs to the case; which rows and columns are kept,
the weights, activations and scores come from the seed.
"""
import math
import random

import torch

from tilesparsity_amd import twgemm as tw
from tilesparsity_amd import twprune

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
_ACTS = {"none": tw.ACT_NONE, "relu": tw.ACT_RELU, "gelu": tw.ACT_GELU}

# rows of A in the first product of a newly built plan (one small evaluation batch)
_FIRST_ROWS = 64

# the convolutions and the first classifier layer of VGG16, K x N as pruning sees them
_VGG16 = ("27x64,576x64,576x128,1152x128,1152x256,2304x256,2304x256,2304x512,4608x512,4608x512,"
          "4608x512,4608x512,4608x512,4096x4096")
# both feed-forward matrices of the twelve encoder layers of BERT-base
_BERT_BASE_FFN = ",".join(["768x3072,3072x768"] * 12)


def listed():
    return [
        # a decoder working off one small beam: one time step of one cell per call, the smallest
        # and most latency-bound call there is
        dict(name="decode_step", kind="lstm", steps=1, M=16, hidden=1024, keep=0.25, G=128, dtype="f16"),
        # the encoder of the NMT model over a sentence batch
        dict(name="nmt_sequence", kind="lstm", steps=50, M=128, hidden=1024, keep=0.25, G=128, dtype="f16"),
        # one request of 128 tokens through a BERT-base feed-forward pair, operands as PyTorch
        # has them (row-major)
        dict(name="bert_base_request", kind="ffn", layout="row", M=128, K=768, N=3072, G=128, keep=0.25,
             dtype="f16"),
        # the same layer pair on a full batch (32 x 128 tokens)
        dict(name="bert_base_batch", kind="ffn", layout="row", M=4096, K=768, N=3072, G=128, keep=0.25,
             dtype="f16"),
        # BERT-large in bfloat16 (16 x 512 tokens), layers chained in the engine's own layout
        dict(name="bert_large_batch", kind="ffn", layout="kmajor", M=8192, K=1024, N=4096, G=128, keep=0.25,
             dtype="bf16"),
        # `test_basic_nn 12800 768 3072 384 1536`: half of the rows, half of the columns
        dict(name="driver_12800", kind="dense", layout="kmajor", M=12800, K=3072, N=768, G=256, keep=0.5,
             keep_cols=0.5, spread=0.0, bias=False, act="none", dtype="f16"),
        # VGG16 conv4_2 as im2col, batch 64: the headline benchmark
        dict(name="conv4_2_batch", kind="dense", layout="kmajor", M=12544, K=4608, N=512, G=128, keep=0.25,
             keep_cols=0.9, spread=0.4, bias=False, act="none", dtype="f16"),
        # conv4_1 for five images with its bias and ReLU: few rows, and not a multiple of 64
        dict(name="conv4_1_five_images", kind="dense", layout="kmajor", M=980, K=2304, N=512, G=128, keep=0.25,
             keep_cols=0.9, spread=0.4, bias=True, act="relu", dtype="f16"),
        # the load-imbalance stress: kept rows from nearly none to nearly all, a tenth of the
        # tiles empty; the largest product
        dict(name="imbalance_stress", kind="dense", layout="kmajor", M=16384, K=4096, N=8192, G=64, keep=0.2,
             keep_cols=0.8, spread=-1.0, bias=False, act="none", dtype="f16"),
        # a pruning step over the feed-forward layers of BERT-base (type 7: rows of tiles)
        dict(name="prune_bert_base", kind="prune", how="1d", layers=_BERT_BASE_FFN, sparsity=75.0, G=128),
        # mixed masks for VGG16: tile-wise plus 5 % of the elements
        dict(name="prune_vgg16_mixed", kind="prune", how="1dmix", layers=_VGG16, sparsity=75.0, G=128),
        # the end of a pruning round on VGG16: masks (columns, then rows), plans, first products
        dict(name="replan_vgg16", kind="replan", layers=_VGG16, sparsity=75.0, G=128, dtype="f16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "ffn", "ffn", "lstm", "prune", "replan"])
    dtype = rng.choice(["f16", "bf16"])
    keep = rng.choice([0.5, 0.25, 0.25, 0.1])
    if kind == "lstm":
        return dict(kind=kind, steps=_log_int(rng, 1, 100), M=_log_int(rng, 1, 256),
                    hidden=rng.choice([256, 512, 1024]), keep=keep, G=128, dtype=dtype)
    if kind in ("prune", "replan"):
        layers, total = [], 0
        most_layers, most = (24, 50_000_000) if kind == "prune" else (12, 30_000_000)
        for _ in range(_log_int(rng, 1, most_layers)):
            k, n = _log_int(rng, 64, 4608), _log_int(rng, 64, 4096)
            if total + k * n <= most:
                layers.append("%dx%d" % (k, n))
                total += k * n
        case = dict(kind=kind, layers=",".join(layers), sparsity=float(rng.randint(40, 92)), G=rng.choice([64, 128]))
        if kind == "prune":
            case["how"] = rng.choice(["1d", "2d", "1dmix"])
        else:
            case["dtype"] = dtype
        return case
    while True:
        M = _log_int(rng, 8, 16384)
        layout = rng.choice(["kmajor", "kmajor", "row"])
        K, N = _log_int(rng, 256, 4608), _log_int(rng, 128, 8192)
        if kind == "ffn":
            N = K * rng.choice([2, 4])
        if layout == "row" or kind == "ffn":  # rows of a row-major matrix start at multiples of 16 bytes
            K, N = K // 8 * 8, N // 8 * 8
        if M * K * N * keep < 1e11 and (K + N) * M < 2e8 and K * N < 4e7:
            break
    case = dict(kind=kind, layout=layout, M=M, K=K, N=N, G=rng.choice([64, 128, 128]), keep=keep, dtype=dtype)
    if kind == "dense":
        case.update(keep_cols=rng.choice([1.0, 1.0, 0.9, 0.8]), spread=rng.choice([0.0, 0.3, 0.4]),
                    bias=rng.random() < 0.6, act=rng.choice(["none", "relu", "gelu"]))
    return case


# ------------------------------------------------------------------------------ weights and plans

def _kept_counts(K, N, G, keep, spread):
    """Kept rows of every tile: keep * K, or uniform within +- spread of that; spread < 0: Beta(0.5, 2)
    with a tenth of the tiles empty."""
    rng = random.Random("%d %d %d %g %g" % (K, N, G, keep, spread))
    counts = []
    for t in range(-(-N // G)):
        if spread < 0:
            counts.append(0 if t % 10 == 9 else int(round(rng.betavariate(0.5, 2.0) * K)))
        else:
            counts.append(min(K, max(1, int(round(K * keep * (1 + rng.uniform(-spread, spread)))))))
    return counts


def _kept_cols(width, keep_cols):
    return max(1, int(round(width * keep_cols)))


def _widths(N, G):
    return [min(G, N - c) for c in range(0, N, G)]


def _weight_elems(K, N, G, keep, keep_cols, spread):
    return sum(k * _kept_cols(w, keep_cols) for k, w in zip(_kept_counts(K, N, G, keep, spread), _widths(N, G)))


def _plan(gen, K, N, G, keep, keep_cols, spread, dtype, std):
    """A plan of random kept rows and columns, built on the device as a pruning run builds it."""
    counts, widths = _kept_counts(K, N, G, keep, spread), _widths(N, G)
    n_tiles = len(counts)
    dev = dict(device="cuda")
    rank = torch.rand((n_tiles, K), generator=gen, **dev).argsort(1).argsort(1)
    rows = rank < torch.tensor(counts, **dev)[:, None]
    key = torch.rand((n_tiles, G), generator=gen, **dev)
    key[-1, widths[-1]:] = 2.0
    cols = key.argsort(1).argsort(1) < torch.tensor([_kept_cols(w, keep_cols) for w in widths], **dev)[:, None]
    mask = rows.t().repeat_interleave(G, 1)[:, :N] & cols.reshape(1, -1)[:, :N]
    mask = mask.to(torch.uint8).contiguous()
    weight = torch.randn((K, N), generator=gen, **dev) * std
    table = [(t * G, w) for t, w in enumerate(widths)]
    return tw.Plan.from_device_mask(K, N, mask.data_ptr(), table, dtype, weight.data_ptr(),
                                    stream=torch.cuda.current_stream().cuda_stream)


def _kmajor(rows, M, dtype):
    """A zeroed K-major matrix of `rows` vectors of M elements, each starting at a multiple of 16 bytes."""
    return torch.zeros((rows, -(-M // 8) * 8), dtype=_DTYPES[dtype], device="cuda")


def _fill(gen, mat, M, relu=False):
    v = torch.randn((mat.shape[0], M), generator=gen, device="cuda")
    mat[:, :M] = v.relu_() if relu else v
    return mat


def _sizes(text):
    return [tuple(int(x) for x in p.split("x")) for p in text.split(",")]


def _scores(gen, sizes):
    """|w| of weights whose rows and columns differ in scale, as trained ones do."""
    out = []
    for k, n in sizes:
        w = torch.randn((k, n), generator=gen, device="cuda").abs_().mul_(math.sqrt(2.0 / k))
        w *= torch.randn((k, 1), generator=gen, device="cuda").mul_(0.3).exp_()
        w *= torch.randn((1, n), generator=gen, device="cuda").mul_(0.3).exp_()
        out.append(w)
    return out


# ------------------------------------------------------------------------------ one pass

def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    kind, s = case["kind"], dict(case)
    if kind in ("prune", "replan"):
        sizes = _sizes(case["layers"])
        s["scores"] = _scores(gen, sizes)
        if kind == "replan":
            s["sizes"], s["plans"] = sizes, []
            s["x"] = [_fill(gen, _kmajor(k, _FIRST_ROWS, case["dtype"]), _FIRST_ROWS, relu=True) for k, n in sizes]
            s["y"] = [_kmajor(n, _FIRST_ROWS, case["dtype"]) for k, n in sizes]
        return s
    M, dtype = case["M"], case["dtype"]
    if kind == "lstm":
        H, T, K = case["hidden"], case["steps"], 2 * case["hidden"]
        s["plan"] = _plan(gen, K, 4 * H, case["G"], case["keep"], 1.0, 0.0, dtype, 0.03)
        s["bias"] = torch.randn(4 * H, generator=gen, device="cuda") * 0.1
        # T + 1 matrices [x_t ; h_(t-1)]: the inputs, and zero for the h before the first step
        s["a"] = torch.zeros((T + 1, K, -(-M // 8) * 8), dtype=_DTYPES[dtype], device="cuda")
        s["a"][:T, :H, :M] = torch.rand((T, H, M), generator=gen, device="cuda") * 2 - 1
        s["c"] = torch.zeros((H, s["a"].shape[2]), device="cuda")
        return s
    K, N, row = case["K"], case["N"], case["layout"] == "row"
    new = (lambda n: torch.zeros((M, n), dtype=_DTYPES[dtype], device="cuda")) if row else (lambda n: _kmajor(n, M, dtype))
    if row:
        s["x"] = torch.randn((M, K), generator=gen, device="cuda").to(_DTYPES[dtype])
    else:
        s["x"] = _fill(gen, _kmajor(K, M, dtype), M, relu=case.get("act") == "relu")
    ffn = kind == "ffn"
    s["plan"] = _plan(gen, K, N, case["G"], case["keep"], case.get("keep_cols", 1.0), case.get("spread", 0.0), dtype,
                      0.02 if ffn else math.sqrt(2.0 / K))
    s["bias1"] = torch.randn(N, generator=gen, device="cuda") * 0.1
    s["y"] = new(N)
    plans = [s["plan"]]
    if ffn:
        s["plan2"] = _plan(gen, N, K, case["G"], case["keep"], 1.0, 0.0, dtype, 0.02)
        s["bias2"] = torch.randn(K, generator=gen, device="cuda") * 0.1
        s["z"] = new(K)
        plans.append(s["plan2"])
    if row:  # a workspace that serves every layer of the program
        need = max(p.staged_workspace(M, tw.ROWMAJOR, tw.ROWMAJOR) for p in plans)
        s["ws"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    return s


def _layer(s, plan, x, y, bias, act, stream):
    layout = tw.ROWMAJOR if s["layout"] == "row" else tw.KMAJOR
    ws = s.get("ws")
    plan.gemm(x.data_ptr(), y.data_ptr(), s["M"], lda=x.shape[1], ldc=y.shape[1], a_layout=layout, c_layout=layout,
              pruned_cols=tw.PRUNED_ZERO if bias is not None else tw.PRUNED_UNTOUCHED, stream=stream,
              bias_ptr=None if bias is None else bias.data_ptr(), activation=act,
              workspace_ptr=None if ws is None else ws.data_ptr(), workspace_bytes=0 if ws is None else ws.numel())


def run(state):
    s, kind = state, state["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "dense":
        _layer(s, s["plan"], s["x"], s["y"], s["bias1"] if s["bias"] else None, _ACTS[s["act"]], stream)
        return s["y"]
    if kind == "ffn":
        _layer(s, s["plan"], s["x"], s["y"], s["bias1"], tw.ACT_GELU, stream)
        _layer(s, s["plan2"], s["y"], s["z"], s["bias2"], tw.ACT_NONE, stream)
        return [s["y"], s["z"]]
    if kind == "lstm":
        a, c, T, H, M = s["a"], s["c"], s["steps"], s["hidden"], s["M"]
        ld = a.shape[2]
        c.zero_()  # a new batch of sequences
        if T == 1:
            s["plan"].lstm_step(a.data_ptr(), M, c.data_ptr(), c.data_ptr(), a[1, H].data_ptr(), lda=ld, ldc_prev=ld,
                                ldc_new=ld, ldh=ld, bias_ptr=s["bias"].data_ptr(), stream=stream)
        else:
            s["plan"].lstm_steps(T, a.data_ptr(), M, c.data_ptr(), lda=ld, ldc=ld, bias_ptr=s["bias"].data_ptr(),
                                 stream=stream)
        return [a[1:, H:], c]
    if kind == "prune":
        fn = {"1d": twprune.tiled_wise_1d, "2d": twprune.tiled_wise_2d, "1dmix": twprune.tiled_wise_1d_mix}[s["how"]]
        return fn(s["scores"], s["sparsity"], s["G"], return_device=True)
    masks, tables = twprune.tiled_wise_2d(s["scores"], s["sparsity"], s["G"], return_device=True, return_tiles=True)
    plans = [tw.Plan.from_device_mask(k, n, m.data_ptr(), table, s["dtype"], w.data_ptr(), stream=stream)
             for (k, n), m, table, w in zip(s["sizes"], masks, tables, s["scores"])]
    for plan, x, y in zip(plans, s["x"], s["y"]):
        plan.gemm(x.data_ptr(), y.data_ptr(), _FIRST_ROWS, pruned_cols=tw.PRUNED_ZERO, stream=stream)
    for old in s["plans"]:  # the round before this one's
        old.destroy()
    s["plans"] = plans
    return [masks, s["y"]]


# ------------------------------------------------------------------------------ what a pass needs

def work(case):
    kind = case["kind"]
    if kind == "lstm":
        M, H, T = case["M"], case["hidden"], case["steps"]
        kept = _weight_elems(2 * H, 4 * H, case["G"], case["keep"], 1.0, 0.0)
        # weight and bias once, x in and h out at every step, the cell state in and out
        return {"bytes": 2 * kept + 16 * H + T * 4 * H * M + 8 * H * M, "flops": 2 * T * M * kept}
    if kind in ("prune", "replan"):
        sizes = _sizes(case["layers"])
        elems = sum(k * n for k, n in sizes)
        if kind == "prune":  # scores in, masks out
            return {"bytes": 5 * elems, "flops": 2 * elems}
        kept = elems * (1 - case["sparsity"] / 100)
        edge = sum(k + n for k, n in sizes) * _FIRST_ROWS
        return {"bytes": 5 * elems + 6 * kept + 2 * edge, "flops": 2 * elems + 2 * _FIRST_ROWS * kept}
    M, K, N = case["M"], case["K"], case["N"]
    w1 = _weight_elems(K, N, case["G"], case["keep"], case.get("keep_cols", 1.0), case.get("spread", 0.0))
    if kind == "ffn":
        w2 = _weight_elems(N, K, case["G"], case["keep"], 1.0, 0.0)
        return {"bytes": 2 * (M * K + w1 + M * N) + 2 * (M * N + w2 + M * K) + 4 * (N + K), "flops": 2 * M * (w1 + w2)}
    cols = N if case["bias"] else sum(_kept_cols(w, case["keep_cols"]) for w in _widths(N, case["G"]))
    return {"bytes": 2 * (M * K + w1 + M * cols), "flops": 2 * M * w1}


def tolerance(case):
    if case["kind"] == "prune":
        return "exact"
    # outputs rounded to 16 bits: 2.1e-4 (f16) and 1.7e-3 (bf16) off the same products in float64,
    # for every kind of case
    return {"rel": 8.5e-4 if case["dtype"] == "f16" else 7e-3}
