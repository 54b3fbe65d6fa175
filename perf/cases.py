"""Performance cases of the bitmap SpMM: what a program that serves a pruned model asks of this framework.

Decode steps (N = 8, 16, 32 columns: one token per sequence of a small batch), batched decode and prefill (N = 64 and
multiples of 128: batch x sequence columns), a chain of decoder layers replayed from a HIP graph, and the device encoder
that compresses weights when a model is loaded.  Sizes are those of the OPT-13B / 30B / 66B linears, plus small and
ragged ones: M and K are multiples of 64 (the group tile), not of the larger blocks a kernel may prefer.
"""
import math

import torch

import spmspm_amd as S
from spmspm_amd.torch_ops import SparseLinearModule

DEVICE = "cuda:0"
GROUP = 64  # rows and columns of a group tile: M and K are multiples of it

# How a linear layer is called.
#   layer    spmspm_amd.SparseLinear, the resident layer object
#   module   SparseLinearModule, the nn.Module around the registered operator
#   abi      SpMM_SplitK_API with the caller's workspace, the library's choice of Split_K
#   noalloc  SpMM_SplitK_API_NoAlloc
#   v3       the 14-argument drop-in call with a Split_K of the caller's (fp16 partial sums)
ENTRIES = ("layer", "module", "abi", "noalloc", "v3")

# The most a drawn case may ask for: the largest listed weight matrix and the largest listed product.
MAX_WEIGHTS = 36864 * 9216
MAX_PRODUCT = 28672 * 7168 * 2048


def linear(name, M, K, N, sparsity, pruning="random", entry="layer", bias=False, act=0, split_k=0):
    return dict(name=name, kind="linear", M=M, K=K, N=N, sparsity=sparsity, pruning=pruning, entry=entry, bias=bias,
                act=act, split_k=split_k)


def listed():
    return [
        # the smallest useful call: a small layer at the smallest batch, launches and host time
        linear("decode_512x1024_n8", 512, 1024, 8, 0.5),
        # OPT-13B output projection in a decode step, as an nn.Module with its bias
        linear("decode_5120x5120_n16", 5120, 5120, 16, 0.6, "magnitude", "module", bias=True),
        # OPT-30B FFN1 in a decode step, the benchmark's headline shape
        linear("decode_28672x7168_n16", 28672, 7168, 16, 0.7),
        # OPT-30B FFN2 at the smallest batch: few rows, long K, deep split
        linear("decode_7168x28672_n8", 7168, 28672, 8, 0.6, entry="abi"),
        # OPT-66B FFN1, the largest weights, at 40 % sparsity and the widest decode batch, bias and ReLU fused
        linear("decode_36864x9216_n32", 36864, 9216, 32, 0.4, bias=True, act=S.ACT_RELU),
        # four OPT-13B decoder layers' linears, recorded once and replayed per token
        dict(name="chain_13b_4layers_n16", kind="chain", D=5120, F=20480, layers=4, N=16, sparsity=0.6,
             pruning="magnitude"),
        # OPT-66B FFN2, batched decode of 64 sequences
        linear("batch_9216x36864_n64", 9216, 36864, 64, 0.4, entry="abi"),
        # OPT-13B FFN1 on a short prompt, bias and ReLU fused
        linear("prefill_20480x5120_n128", 20480, 5120, 128, 0.6, "magnitude", "module", bias=True, act=S.ACT_RELU),
        # a ragged matrix (65 row blocks, 77 k blocks) through the drop-in call with the caller's split
        linear("prefill_4160x4928_n384", 4160, 4928, 384, 0.5, entry="v3", split_k=2),
        # OPT-30B FFN1 on a full prompt (or a batch of them)
        linear("prefill_28672x7168_n2048", 28672, 7168, 2048, 0.7),
        # model load: a large matrix encoded in one pass over W
        dict(name="encode_28672x7168_onepass", kind="encode", form="onepass", M=28672, K=7168, sparsity=0.7,
             pruning="random"),
        # model load: an ordinary matrix through the two-call encoder, which allocates exactly
        dict(name="encode_5120x5120_twocall", kind="encode", form="twocall", M=5120, K=5120, sparsity=0.6,
             pruning="magnitude"),
    ]


def _blocks(rng, lo, hi):
    """A multiple of 64, spread over the logarithm of lo..hi, any count of blocks (odd ones included)."""
    return GROUP * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / GROUP))


def draw(rng):
    kind = rng.choices(("decode", "prefill", "chain", "encode"), (9, 7, 1, 3))[0]
    sparsity = round(rng.uniform(0.4, 0.8), 2)
    pruning = rng.choice(("random", "magnitude"))
    if kind == "chain":
        D = _blocks(rng, 1024, 7168)
        return dict(kind="chain", D=D, F=4 * D, layers=rng.randint(2, 4), N=rng.choice((8, 16, 32)), sparsity=sparsity,
                    pruning=pruning)
    while True:
        M, K = _blocks(rng, 512, 36864), _blocks(rng, 512, 36864)
        if M * K <= MAX_WEIGHTS:
            break
    if kind == "encode":
        return dict(kind="encode", form=rng.choice(("onepass", "twocall")), M=M, K=K, sparsity=sparsity, pruning=pruning)
    if kind == "decode":
        N = rng.choice((8, 16, 32))
    else:
        top = max(1, min(2048, MAX_PRODUCT // (M * K)) // 128)
        N = 64 if rng.random() < 0.25 else 128 * max(1, round(math.exp(rng.uniform(0.0, math.log(top)))))
    entry = rng.choice(ENTRIES)
    fused = entry in ("layer", "module") and rng.random() < 0.5
    return dict(kind="linear", M=M, K=K, N=N, sparsity=sparsity, pruning=pruning, entry=entry, bias=fused,
                act=rng.choice((S.ACT_NONE, S.ACT_RELU, S.ACT_GELU)) if fused else S.ACT_NONE,
                split_k=rng.randint(1, 4) if entry == "v3" else 0)


def _weight(gen, M, K, sparsity, pruning):
    """fp16 N(0, 0.02), pruned by a random mask or by magnitude (the threshold that prunes `sparsity` of a normal)."""
    W = torch.empty((M, K), dtype=torch.float16, device=DEVICE)
    below = 0.02 * math.sqrt(2.0) * float(torch.erfinv(torch.tensor(sparsity, dtype=torch.float64)))
    rows = max(1, (1 << 25) // K)
    for r in range(0, M, rows):
        w = torch.randn((min(rows, M - r), K), generator=gen, device=DEVICE) * 0.02
        drop = w.abs() < below if pruning == "magnitude" else torch.rand(w.shape, generator=gen, device=DEVICE) < sparsity
        W[r:r + rows] = w.masked_fill_(drop, 0.0)
    return W


def _with_value_count(W, total):
    """W with as few further entries zeroed as leave `total` encoded values (a multiple of 8): an encoding's arrays then
    have one size whatever the seed.  Eight non-zeros fewer in a group tile are eight encoded values fewer, since every
    group tile's run is padded to a multiple of eight; the removals are dealt evenly over the group tiles."""
    M, K = W.shape
    tiles = W.view(M // GROUP, GROUP, K // GROUP, GROUP).transpose(1, 2)
    count = (tiles != 0).sum(dim=(2, 3)).view(-1)
    excess = (int((count + 7).div(8, rounding_mode="floor").sum()) * 8 - total) // 8
    share = excess // count.numel() + (torch.arange(count.numel(), device=W.device) < excess % count.numel())
    for gm in range(M // GROUP):
        block = tiles[gm].reshape(K // GROUP, GROUP * GROUP)
        drop = (block != 0).cumsum(1) <= 8 * share[gm * (K // GROUP):(gm + 1) * (K // GROUP), None]
        tiles[gm] = block.masked_fill(drop, 0.0).view(K // GROUP, GROUP, GROUP)
    return W


def _activations(gen, N, K):
    return (torch.rand((N, K), generator=gen, device=DEVICE) * 2 - 1).half()


def _encoded(gen, M, K, sparsity, pruning):
    return S.InitSparseMatrixA_bitmap_device(_weight(gen, M, K, sparsity, pruning))


def _layer(M, K, arrays, bias=None, act=S.ACT_NONE):
    values, bitmaps, offsets = arrays
    none = torch.empty(0, dtype=torch.int32).numpy()
    comp = S.CompressedMatrix(M=M, K=K, num_gtiles=offsets.numel() - 1, values=values.cpu().numpy().view("u2"),
                              tile_counts=none, median=none, offsets=offsets.cpu().numpy(),
                              bitmaps=bitmaps.cpu().numpy().view("u8"), max_nnz=0)
    return S.SparseLinear(comp, device=DEVICE, bias=bias, activation=act)


def _prepare_linear(case, gen):
    M, K, N, entry = case["M"], case["K"], case["N"], case["entry"]
    arrays = _encoded(gen, M, K, case["sparsity"], case["pruning"])
    x = _activations(gen, N, K)
    bias = (torch.rand(M, generator=gen, device=DEVICE) - 0.5).half() if case["bias"] else None
    state = dict(case, arrays=arrays, x=x)
    if entry == "layer":
        state["call"] = _layer(M, K, arrays, bias, case["act"])
    elif entry == "module":
        state["call"] = SparseLinearModule(M, K, *arrays, bias=bias, activation=case["act"])
    else:
        state["out"] = torch.empty((N, M), dtype=torch.float16, device=DEVICE)
        if entry == "abi":
            need = S.SpMM_WorkspaceBytes(M, N, K, 0)
        else:  # v3: room for split_k slabs of fp16 partial sums
            need = 2 * M * N * case["split_k"] if entry == "v3" else 0
        state["ws"] = torch.empty(need, dtype=torch.uint8, device=DEVICE) if need else None
    return state


def _prepare_chain(case, gen):
    """`layers` x {QKV, output projection, FFN1 with ReLU, FFN2} with weights of their own.  The attention between QKV
    and the output projection is not part of this framework: its result is a fixed input of every layer."""
    D, F, N = case["D"], case["F"], case["N"]

    def lin(M, K, act=S.ACT_NONE):
        arrays = _encoded(gen, M, K, case["sparsity"], case["pruning"])
        bias = (torch.rand(M, generator=gen, device=DEVICE) - 0.5).half()
        return _layer(M, K, arrays, bias, act)

    steps, x = [], _activations(gen, N, D)
    new = lambda m: torch.empty((N, m), dtype=torch.float16, device=DEVICE)
    h = x
    for _ in range(case["layers"]):
        qkv, proj, ffn1, ffn2 = lin(3 * D, D), lin(D, D), lin(F, D, S.ACT_RELU), lin(D, F)
        attended = _activations(gen, N, D)
        a, b, c, d = new(3 * D), new(D), new(F), new(D)
        steps += [(qkv, h, a), (proj, attended, b), (ffn1, b, c), (ffn2, c, d)]
        h = d

    def once():
        for layer, inp, out in steps:
            layer(inp, out=out)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        once()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        once()
    return dict(case, steps=steps, graph=graph, outs=[out for _, _, out in steps])


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    if case["kind"] == "linear":
        return _prepare_linear(case, gen)
    if case["kind"] == "chain":
        return _prepare_chain(case, gen)
    M, K = case["M"], case["K"]
    W = _weight(gen, M, K, case["sparsity"], case["pruning"])
    # six standard deviations of the count below its mean
    kept = (1 - case["sparsity"]) * M * K
    return dict(case, W=_with_value_count(W, int(kept - 6 * math.sqrt(case["sparsity"] * kept)) // 8 * 8))


def run(s):
    if s["kind"] == "chain":
        s["graph"].replay()
        return s["outs"]
    if s["kind"] == "encode":
        encode = S.InitSparseMatrixA_bitmap_device_onepass if s["form"] == "onepass" else S.InitSparseMatrixA_bitmap_device
        return encode(s["W"])
    if s["entry"] in ("layer", "module"):
        return s["call"](s["x"])
    values, bitmaps, offsets = s["arrays"]
    M, N, K = s["M"], s["N"], s["K"]
    if s["entry"] == "abi":
        err = S.SpMM_SplitK_API(None, values, bitmaps, offsets, s["x"], s["out"], M, N, K, s["ws"], 0)
    elif s["entry"] == "noalloc":
        err = S.SpMM_SplitK_API_NoAlloc(None, values, bitmaps, offsets, s["x"], s["out"], M, N, K, 0)
    else:
        err = S.SpMM_SplitK_API_bitmap_v3(None, None, values, offsets, None, bitmaps, None, s["x"], s["out"], M, N, K,
                                          s["ws"], s["split_k"])
    if err:
        raise RuntimeError(f"the library returned hipError_t {err}")
    return s["out"]


def exact(case, seed):
    """What `run` returns for these inputs in float64: the dense weights, no rounding between the layers of a chain.  The
    inputs are drawn in the order in which `prepare` draws them.  An encoding is whole numbers and has none."""
    if case["kind"] == "encode":
        return None
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def weight(M, K):
        return _weight(gen, M, K, case["sparsity"], case["pruning"])

    def bias(M):
        return (torch.rand(M, generator=gen, device=DEVICE) - 0.5).half().double()

    def product(x, W, b, act):
        y = x @ W.double().t()
        if b is not None:
            y += b
        if act == S.ACT_RELU:
            y = y.relu()
        elif act == S.ACT_GELU:
            y = torch.nn.functional.gelu(y, approximate="tanh")
        return y

    if case["kind"] == "linear":
        W = weight(case["M"], case["K"])
        x = _activations(gen, case["N"], case["K"]).double()
        return product(x, W, bias(case["M"]) if case["bias"] else None, case["act"])
    D, F, N = case["D"], case["F"], case["N"]
    outs, h = [], _activations(gen, N, D).double()
    for _ in range(case["layers"]):
        linears = []
        for M, K, act in ((3 * D, D, S.ACT_NONE), (D, D, S.ACT_NONE), (F, D, S.ACT_RELU), (D, F, S.ACT_NONE)):
            W = weight(M, K)
            linears.append((W, bias(M), act))
        attended = _activations(gen, N, D).double()
        qkv, proj, ffn1, ffn2 = linears
        a = product(h, *qkv)
        b = product(attended, *proj)
        c = product(b, *ffn1)
        h = product(c, *ffn2)
        outs += [a, b, c, h]
    return outs


def _weight_bytes(M, K, sparsity):
    """Compressed arrays of one matrix: fp16 values, one 64-bit bitmap per 8x8 tile, one offset per group tile."""
    return 2 * (1 - sparsity) * M * K + M * K / 8 + 4 * (M * K // 4096 + 1)


def work(case):
    if case["kind"] == "encode":
        M, K = case["M"], case["K"]
        return {"bytes": 2 * M * K + _weight_bytes(M, K, case["sparsity"]), "flops": 0}
    N = case["N"]
    if case["kind"] == "chain":
        D, F = case["D"], case["F"]
        shapes = [(3 * D, D), (D, D), (F, D), (D, F)] * case["layers"]
    else:
        shapes = [(case["M"], case["K"])]
    # flops of the dense product: the matrix cores multiply the zeros too
    return {"bytes": sum(_weight_bytes(M, K, case["sparsity"]) + 2 * N * (M + K) for M, K in shapes),
            "flops": sum(2 * M * K * N for M, K in shapes)}


def tolerance(case):
    """Four times the distance from a float64 product of the same inputs, as measured over the listed cases and thirty
    drawn ones: 2.1e-4 for one fp16 rounding of an fp32 sum (largest single difference 4.9e-4 of the value), 3.1e-4 and
    1.9e-3 where the caller's split adds fp16 partial sums, 4.1e-4 and 1.7e-3 at the end of a chain of layers (four
    products in a row between two attention inputs)."""
    if case["kind"] == "encode":
        return "exact"
    if case["kind"] == "chain":
        return {"rel": 1.6e-3, "max": 7e-3}
    if case["entry"] == "v3" and case["split_k"] > 1:
        return {"rel": 1.2e-3, "max": 7.5e-3}
    return {"rel": 8.5e-4, "max": 2e-3}
