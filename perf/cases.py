"""The work that users of this framework have it do, as cases that can be timed and compared.

Four kinds of case, each through the entry points a program would call:

* `linear`: one quantized projection of fp16 rows, `programs.QuantizedLinear.run` (A8 quantiser + projection);
* `layer`: the quantized projections of one decoder layer with what produces their int8 rows, eight `lib.Kernel`
  launches (seven for one row); at decode sizes captured once and replayed, as an engine does with its decode step;
* `moe`: one routed-expert layer, `programs.MoeLayer.run`;
* `token`: the same expert layer for a single token, `programs.MoeTokenLayer.run`.
"""
import math

import numpy as np
import torch

from orinfer_amd import codebook, lib, programs

BOOK_BYTES = 1024
GRAPH_ROWS = 64        # decode batches up to this many rows are replayed from a graph
LARGEST_MATRIX = 34816 * 5120
LARGEST_BANK = 128 * 2048 * 512


def listed():
    return [
        # the smallest call there is: one decode row through one small projection, launched eagerly
        {"name": "linear q4 1 row", "kind": "linear", "codec": "q4", "rows": 1, "n": 9728, "k": 2560, "packed_k": 0},
        # a batch of decoding requests through a wide projection in the stored (K-major) layout
        {"name": "linear q4 8 rows", "kind": "linear", "codec": "q4", "rows": 8, "n": 17408, "k": 5120, "packed_k": 128},
        # the int8 down projection of such a layer for a larger decode batch: few channels, long rows
        {"name": "linear w8 24 rows", "kind": "linear", "codec": "w8", "rows": 24, "n": 5120, "k": 17408, "packed_k": 0},
        # a short prompt of ragged length through the attention input projection
        {"name": "linear q4 200 rows", "kind": "linear", "codec": "q4", "rows": 200, "n": 7168, "k": 5120, "packed_k": 128},
        # one prefill chunk of the usual length
        {"name": "linear q4 512 rows", "kind": "linear", "codec": "q4", "rows": 512, "n": 17408, "k": 5120, "packed_k": 0},
        # an int8 projection of a long prompt
        {"name": "linear w8 8192 rows", "kind": "linear", "codec": "w8", "rows": 8192, "n": 4096, "k": 4096, "packed_k": 0},
        # one decode step of a 27B-class layer, replayed from a graph: single request, then a batch of requests
        {"name": "layer 1 row", "kind": "layer", "rows": 1, "hidden": 5120, "qkv": 7168, "inner": 17408},
        {"name": "layer 20 rows", "kind": "layer", "rows": 20, "hidden": 5120, "qkv": 7168, "inner": 17408},
        # the same layer over a long prompt
        {"name": "layer 8192 rows", "kind": "layer", "rows": 8192, "hidden": 5120, "qkv": 7168, "inner": 17408},
        # routed experts: single-token decode, a decode batch (or short prompt), a long prompt
        {"name": "moe 1 token", "kind": "token", "experts": 128, "top_k": 8, "hidden": 2048, "inner": 512},
        {"name": "moe 256 tokens", "kind": "moe", "tokens": 256, "experts": 128, "top_k": 8, "hidden": 2048, "inner": 512},
        {"name": "moe 4096 tokens", "kind": "moe", "tokens": 4096, "experts": 128, "top_k": 8, "hidden": 2048, "inner": 512},
    ]


def _spread(rng, low, high, step=1):
    """A whole multiple of `step` in [low, high], spread evenly over the logarithm."""
    value = math.exp(rng.uniform(math.log(low), math.log(high + 1)))
    return min(high, max(low, int(value) // step * step))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "layer", "layer", "moe", "moe", "token"))
    if kind == "linear":
        codec = rng.choice(("q4", "q4", "w8"))
        k = _spread(rng, 1024, 17408, 128)
        n = _spread(rng, 1024, min(34816, LARGEST_MATRIX // k), 16)
        packed_k = rng.choice((0, 128)) if codec == "q4" else 0
        return {"kind": kind, "codec": codec, "rows": _spread(rng, 1, 8192), "n": n, "k": k, "packed_k": packed_k}
    if kind == "layer":
        hidden = _spread(rng, 1024, 5120, 256)
        return {"kind": kind, "rows": _spread(rng, 1, 8192), "hidden": hidden,
                "qkv": _spread(rng, hidden, 7168 * hidden // 5120, 128), "inner": _spread(rng, 2 * hidden, 17 * hidden // 5, 256)}
    experts = rng.choice((16, 32, 64, 128))
    hidden = _spread(rng, 1024, 4096, 128)
    shape = {"experts": experts, "top_k": rng.choice((2, 4, 6, 8)), "hidden": hidden,
             "inner": _spread(rng, 256, min(1536, LARGEST_BANK // (experts * hidden)), 128)}
    return dict({"kind": "moe", "tokens": _spread(rng, 2, 4096)} if kind == "moe" else {"kind": "token"}, **shape)


def prepare(case, seed):
    return {"linear": _Linear, "layer": _Layer, "moe": _Moe, "token": _Token}[case["kind"]](case, seed)


def run(state):
    return state.run()


class _Source:
    """Seeded inputs: weights on the host as a loader has them, activations on the GPU."""

    def __init__(self, seed):
        self.host = np.random.default_rng(seed)
        self.gpu = torch.Generator(device="cuda").manual_seed(int(seed))

    def codes(self, shape, dtype):
        """Uniform lattice codes (u32: two-stage, u16: single-stage)."""
        count = math.prod(shape) * np.dtype(dtype).itemsize
        return np.frombuffer(self.host.bytes(count), dtype).reshape(shape)

    def int8(self, shape):
        """int8 weights, the -128 that a symmetric quantiser never writes left out."""
        return np.maximum(np.frombuffer(self.host.bytes(math.prod(shape)), np.int8), -127).reshape(shape)

    def scales(self, shape, codec, k):
        """Channel scales that keep the variance of a row, as trained weights roughly do."""
        rms = {"q4": 22.0, "q2": 5.4, "w8": 73.0}[codec]
        unit = 1.0 / (rms * math.sqrt(k))
        return self.host.uniform(0.5 * unit, 1.5 * unit, shape).astype(np.float16)

    def normal(self, *shape, dtype=torch.float16):
        return torch.randn(shape, generator=self.gpu, device="cuda", dtype=torch.float32).to(dtype)

    def activations(self, rows, k):
        """fp16 rows ~N(0,1) with one channel in a thousand twenty times as large."""
        x = self.normal(rows, k, dtype=torch.float32)
        x[:, torch.randperm(k, generator=self.gpu, device="cuda")[: max(1, k // 1000)]] *= 20.0
        return x.half()

    def signs(self, k):
        return torch.randint(0, 2, (k,), generator=self.gpu, device="cuda", dtype=torch.int8) * 2 - 1

    def logits(self, tokens, experts):
        """Router logits with a Zipf(1.1) preference over a random order of the experts."""
        rank = torch.randperm(experts, generator=self.gpu, device="cuda") + 1
        return self.normal(tokens, experts, dtype=torch.float32) - 1.1 * rank.float().log()


class _Linear:
    def __init__(self, case, seed):
        source = _Source(seed)
        codec, n, k = case["codec"], case["n"], case["k"]
        weight = source.codes((n, k // 8), np.uint32) if codec == "q4" else source.int8((n, k))
        self.linear = programs.QuantizedLinear(codec, weight, source.scales(n, codec, k), max(512, case["rows"]),
                                               packed_k=case["packed_k"])
        self.x = source.activations(case["rows"], k)

    def run(self):
        return self.linear.run(self.x)


class _Layer:
    """RMSNorm + rotation + A8 -> qkv; rotation + A8 -> output projection; RMSNorm + rotation + A8 -> gate | up;
    SwiGLU + A8 -> down (int8).  Attention itself is not the framework's: its output is an input here."""

    def __init__(self, case, seed):
        rows, hidden, qkv, inner = self.rows, self.hidden, self.n_qkv, self.inner = (
            case["rows"], case["hidden"], case["qkv"], case["inner"])
        source = _Source(seed)
        f16, f32, i8 = (dict(dtype=d, device="cuda") for d in (torch.float16, torch.float32, torch.int8))
        self.x, self.attention = source.activations(rows, hidden), source.normal(rows, hidden)
        self.residual = source.normal(rows, hidden, dtype=torch.float32)
        self.norm = [source.normal(hidden) * 0.1 for _ in range(2)]
        self.signs = [source.signs(hidden) for _ in range(3)]
        self.book = self._device(codebook.book())
        self.projections = {}
        for name, n, k in (("qkv", qkv, hidden), ("o", hidden, hidden), ("gate_up", 2 * inner, hidden)):
            kernel = lib.Kernel("e8p_q4_projection", M=rows, N=n, K=k, dynamic_rows=True, packed_k=128, workspace=True)
            self.projections[name] = (kernel, dict(Book=self.book, W=self._device(source.codes((k // 128, n, 16), np.uint32)),
                                                   S=self._device(source.scales(n, "q4", k)), Workspace=kernel.workspace()))
        self.down = lib.Kernel("int8_projection", M=rows, N=hidden, K=inner, dynamic_rows=True, workspace=True)
        self.down_buffers = dict(Weight=self._device(source.int8((hidden, inner))),
                                 WeightScale=self._device(source.scales(hidden, "w8", inner)), Workspace=self.down.workspace())
        self.normed = lib.Kernel("residual_norm_rotate_a8", M=rows, K=hidden)
        self.rotated = lib.Kernel("rotate_activation_a8", M=rows, K=hidden)
        self.activated = lib.Kernel("activation_quantization", K=inner, fused=True)
        # one row: the projection rotates and quantises its fp16 row itself
        self.o_fused = rows == 1 and lib.Kernel("e8p_q4_projection", M=1, N=hidden, K=hidden, packed_k=128,
                                                input_dtype="float16", rotate=True)
        self.codes, self.scale = torch.empty((rows, hidden), **i8), torch.empty((rows,), **f16)
        self.y = torch.empty((rows, hidden), **f16)
        self.sums = [torch.empty((rows, hidden), **f32) for _ in range(2)]
        self.out = {n: torch.empty((rows, w), **f16) for n, w in
                    (("qkv", qkv), ("o", hidden), ("gate_up", 2 * inner), ("down", hidden))}
        self.act_codes, self.act_scale = torch.empty((rows, inner), **i8), torch.empty((rows, 1), **f16)
        self.graph = None
        if rows <= GRAPH_ROWS:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                self.enqueue(side.cuda_stream)
            side.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph, stream=side):
                self.enqueue(side.cuda_stream)

    @staticmethod
    def _device(array):
        view = {np.dtype(np.uint32): np.int32}.get(array.dtype, array.dtype)
        return torch.from_numpy(np.array(array).view(view)).cuda()

    def enqueue(self, stream):
        def norm(i, x, residual):
            self.normed(stream=stream, Q=self.codes, R=residual, RO=self.sums[i], S=self.scale, Signs=self.signs[i],
                        W=self.norm[i], X=x, Y=self.y)

        def project(name):
            kernel, buffers = self.projections[name]
            kernel(stream=stream, A=self.codes, AS=self.scale, Out=self.out[name], m=self.rows, **buffers)

        norm(0, self.x, self.residual)
        project("qkv")
        if self.o_fused:
            weights = self.projections["o"][1]
            self.o_fused(stream=stream, A=self.attention, AS=self.scale, Book=self.book, Out=self.out["o"], S=weights["S"],
                         Signs=self.signs[2], W=weights["W"])
        else:
            self.rotated(stream=stream, Q=self.codes, S=self.scale, Signs=self.signs[2], X=self.attention)
            project("o")
        norm(1, self.out["o"], self.sums[0])
        project("gate_up")
        self.activated(stream=stream, Mask=None, Q=self.act_codes, S=self.act_scale, X=self.out["gate_up"], rows=self.rows)
        self.down(stream=stream, A=self.act_codes, Output=self.out["down"], TokenScale=self.act_scale, m=self.rows,
                  **self.down_buffers)

    def run(self):
        if self.graph is not None:
            self.graph.replay()
        else:
            self.enqueue(torch.cuda.current_stream().cuda_stream)
        return dict(self.out, residual=self.sums[1])


def _bank(case, source):
    experts, hidden, inner = case["experts"], case["hidden"], case["inner"]
    return (source.codes((experts, 2 * inner, hidden // 8), np.uint16), source.scales((experts, 2 * inner), "q2", hidden),
            source.codes((experts, hidden, inner // 8), np.uint16), source.scales((experts, hidden), "q2", inner))


class _Moe:
    def __init__(self, case, seed):
        source = _Source(seed)
        tokens, experts, hidden = case["tokens"], case["experts"], case["hidden"]
        self.layer = programs.MoeLayer(tokens, experts, case["top_k"], hidden, case["inner"], *_bank(case, source))
        self.x, self.logits = source.normal(tokens, hidden), source.logits(tokens, experts)

    def run(self):
        return self.layer.run(self.x, self.logits)


class _Token:
    def __init__(self, case, seed):
        source = _Source(seed)
        self.layer = programs.MoeTokenLayer(case["experts"], case["top_k"], case["hidden"], case["inner"], *_bank(case, source))
        self.x, self.logits = source.normal(1, case["hidden"]), source.logits(1, case["experts"])

    def run(self):
        return self.layer.run(self.x, self.logits)


def _experts_touched(tokens, experts, top_k):
    """Experts that a batch of this size reaches with the logits of `_Source.logits` (one fixed drawing)."""
    logits = np.random.default_rng(0).standard_normal((tokens, experts)) - 1.1 * np.log(np.arange(1, experts + 1))
    return len(np.unique(np.argpartition(-logits, top_k - 1, axis=1)[:, :top_k]))


def work(case):
    """Weights, inputs and outputs once each; int8 rows and everything else in between need not touch memory."""
    kind = case["kind"]
    if kind == "linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        weight = n * k // 2 + BOOK_BYTES if case["codec"] == "q4" else n * k
        return {"bytes": weight + 2 * n + 2 * rows * (n + k), "flops": 2 * rows * n * k}
    if kind == "layer":
        rows, hidden, qkv, inner = case["rows"], case["hidden"], case["qkv"], case["inner"]
        q4 = (qkv + hidden + 2 * inner) * hidden
        outputs = 2 * (qkv + 2 * hidden + 2 * inner) + 4 * hidden  # the projections, the second residual sum
        inputs = 2 * 2 * hidden + 4 * hidden                       # layer input, attention output, residual
        return {"bytes": q4 // 2 + hidden * inner + rows * (inputs + outputs), "flops": 2 * rows * (q4 + hidden * inner)}
    tokens, top_k, hidden, inner = case.get("tokens", 1), case["top_k"], case["hidden"], case["inner"]
    touched = _experts_touched(tokens, case["experts"], top_k)
    return {"bytes": touched * (3 * hidden * inner // 4 + 2 * (hidden + 2 * inner)) + tokens * 4 * (hidden + case["experts"]),
            "flops": 6 * tokens * top_k * hidden * inner}


def tolerance(case):
    # A projection of fp16 rows is defined to the bit: A8 codes, int32 sums, two fp32 products, one cast.
    if case["kind"] == "linear":
        return "exact"
    # The order of the RMSNorm's fp32 sum and exp() in SwiGLU may move an fp16 value by one ulp and, where that lies at a
    # rounding boundary, an A8 code by one of about thirty steps rms; fp16 outputs add 3e-4 of their own.
    return {"rel": 3e-3}
