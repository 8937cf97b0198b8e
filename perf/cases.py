"""The work that programs written against this package have it do, as measurable cases.

Every case is one step of such a program through the public API (``nb.compile``,
``nb.value_and_grad``, ``nb.realize_all``, ``nb.nn``, ``nb.ops``): gradients, updated parameters or
logits come back whole.  ``listed()`` holds one case per kind of use over the range from the
smallest calls, which are all latency, to the largest; ``draw()`` gives further cases of the same
kinds and ranges.  The step functions are compiled once per program, as a user's are; what a case
prepares is data: inputs, parameters and optimizer state on the GPU.
"""
from __future__ import annotations

import functools
import math

import torch

import nabla_amd as nb

F = nb.nn.functional

NF4_LEVELS = nb.nn.finetune.qlora.NF4_CODEBOOK


# ---- the cases ------------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # a first network on a table of 200 points, evaluated eagerly (the default mode) with
        # AdamW: every pass records, looks up and launches a handful of tiny kernels
        dict(name="mlp_toy_eager", kind="mlp", batch=200, width_in=4, hidden=32, width_out=1, depth=1,
             optimizer=True, compiled=False),
        # the two-layer perceptron on image-sized rows, compiled: launch-bound
        dict(name="mlp_compiled", kind="mlp", batch=128, width_in=784, hidden=256, width_out=10, depth=1,
             optimizer=False, compiled=True),
        # the fused elementwise + reduction chain at its full size: memory-bound
        dict(name="chain_8192", kind="chain", rows=8192, cols=8192, dtype="float32"),
        # a row program of a user's own (normalise, gate, softmax) on rows of no round size
        dict(name="rows_ragged", kind="rows", rows=6001, cols=1003, dtype="float32"),
        # one pre-norm transformer block at training size
        dict(name="block_train", kind="block", batch=8, seq=1024, width=1024, heads=16, ff=4096,
             dtype="bfloat16", causal=True, dropout=0.0, optimizer=False),
        # the same with sequences as data has them: no multiple of a tile, attention both ways
        dict(name="block_ragged_seq", kind="block", batch=6, seq=333, width=512, heads=8, ff=2048,
             dtype="bfloat16", causal=False, dropout=0.0, optimizer=False),
        # a layer trained with the package's defaults: float32, dropout 0.1, AdamW in the step
        dict(name="block_f32_dropout", kind="block", batch=4, seq=256, width=512, heads=8, ff=2048,
             dtype="float32", causal=True, dropout=0.1, optimizer=True),
        # scoring a prompt: forward only through a small decoder, logits of every position
        dict(name="decoder_logits", kind="decoder", layers=4, batch=1, seq=1800, width=1024, heads=8, ff=4096,
             vocab=32000),
        # the convolutional network's training step
        dict(name="cnn_train", kind="cnn", batch=64, hw=32, c0=3, c1=64, c2=128, c3=256, classes=10, train=True),
        # classifying a batch of grey 28 x 28 images: forward only, channels of no round size
        dict(name="cnn_classify", kind="cnn", batch=50, hw=28, c0=1, c1=24, c2=40, c3=72, classes=10, train=False),
        # adapters on a decoder of twelve layers: the largest step
        dict(name="lora_train", kind="lora", layers=12, batch=4, seq=2048, width=2048, heads=16, ff=8192,
             vocab=32000, rank=16),
        # adapters on a feed-forward pair whose frozen weights are four-bit codes
        dict(name="qlora_train", kind="qlora", tokens=1000, width=1024, ff=4096, rank=8),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["mlp", "mlp", "chain", "rows", "block", "block", "decoder", "cnn", "cnn", "lora", "qlora"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 8, 4096), width_in=_log(rng, 2, 1024), hidden=_log(rng, 16, 1024),
                    width_out=_log(rng, 1, 128), depth=rng.randint(1, 4), optimizer=rng.random() < 0.5,
                    compiled=rng.random() < 0.5)
    if kind in ("chain", "rows"):
        cols = _log(rng, 48, 16384)
        return dict(kind=kind, rows=_log(rng, 32, min(1 << 16, (1 << 26) // cols)), cols=cols,
                    dtype=rng.choice(["float32", "bfloat16"]))
    if kind == "block":
        head, heads = rng.choice([(32, 8), (64, 4), (64, 8), (64, 16), (128, 4), (128, 8)])
        batch = rng.randint(1, 8)
        seq = _log(rng, 48, 1024)
        if rng.random() < 0.4:
            seq = max(128, seq // 128 * 128)
        optimizer = rng.random() < 0.5
        return dict(kind=kind, batch=batch, seq=seq, width=head * heads, heads=heads, ff=4 * head * heads,
                    dtype=rng.choice(["bfloat16", "bfloat16", "float32"]), causal=rng.random() < 0.5,
                    dropout=0.1 if optimizer and rng.random() < 0.5 else 0.0, optimizer=optimizer)
    if kind == "decoder":
        width = rng.choice([512, 1024, 2048])
        return dict(kind=kind, layers=rng.randint(1, 6), batch=rng.randint(1, 3), seq=_log(rng, 40, 2048),
                    width=width, heads=width // rng.choice([64, 128]), ff=4 * width, vocab=_log(rng, 1000, 32000))
    if kind == "cnn":
        return dict(kind=kind, batch=_log(rng, 1, 96), hw=2 * rng.randint(7, 20), c0=rng.choice([1, 3]),
                    c1=8 * rng.randint(2, 8), c2=8 * rng.randint(3, 16), c3=8 * rng.randint(4, 32),
                    classes=_log(rng, 2, 100), train=rng.random() < 0.6)
    if kind == "lora":
        width = rng.choice([512, 1024, 2048])
        return dict(kind=kind, layers=rng.randint(1, 6), batch=rng.randint(1, 4), seq=64 * _log(rng, 2, 32),
                    width=width, heads=width // rng.choice([64, 128]), ff=4 * width, vocab=_log(rng, 1000, 32000),
                    rank=rng.choice([4, 8, 16, 32]))
    return dict(kind=kind, tokens=_log(rng, 16, 8192), width=64 * rng.randint(4, 32), ff=64 * rng.randint(8, 64),
                rank=rng.choice([4, 8, 16, 32]))


# ---- the programs ------------------------------------------------------------------------------
def _mlp_loss(params, x, y):
    h = x
    for w, b in params[:-1]:
        h = nb.relu(h @ w + b)
    w, b = params[-1]
    return F.mse_loss(h @ w + b, y)


def _adamw(params, grads, opt):
    return nb.nn.optim.adamw_update(params, grads, opt, lr=1e-3, weight_decay=0.01, realize=False)


def _mlp_step(params, x, y):
    return nb.value_and_grad(_mlp_loss)(params, x, y)


def _mlp_update(params, opt, x, y):
    loss, grads = nb.value_and_grad(_mlp_loss)(params, x, y)
    return loss, *_adamw(params, grads, opt)


def _chain(x, y):
    p = x * y
    m = nb.reduce_max(p, axis=1, keepdims=True)
    return nb.reduce_sum(nb.exp(p - m) * nb.relu(x), axis=1)


@nb.compile
def _chain_step(x, y):
    return _chain(x, y), nb.grad(lambda a, b: nb.reduce_sum(_chain(a, b)))(x, y)


def _rows(x, gate, weight, bias):
    h = F.layer_norm(x, weight, bias)
    return nb.softmax(h * nb.silu(gate) + x, axis=-1)


@nb.compile
def _rows_step(x, gate, weight, bias, target):
    def loss(x, gate):
        err = _rows(x, gate, weight, bias) - target
        return nb.reduce_sum(err * err)

    return nb.value_and_grad(loss, argnums=(0, 1))(x, gate)


def _heads(t, batch, seq, heads):
    return nb.swap_axes(nb.reshape(t, (batch, seq, heads, int(t.shape[-1]) // heads)), 1, 2)


def _block(x, p, heads, causal, dropout=0.0, lora=None):
    """A pre-norm transformer block.  The key projection has no bias: a softmax does not see one,
    so its gradient would be nothing but rounding."""
    b, s, d = (int(n) for n in x.shape)
    h = F.layer_norm(x, p["ln1_w"], p["ln1_b"])
    if lora is None:
        q, v = h @ p["wq"], h @ p["wv"]
    else:
        q = nb.nn.finetune.lora_linear(h, p["wq"], lora["q"], alpha=16.0)
        v = nb.nn.finetune.lora_linear(h, p["wv"], lora["v"], alpha=16.0)
    q, k, v = q + p["bq"], h @ p["wk"], v + p["bv"]
    a = F.scaled_dot_product_attention(_heads(q, b, s, heads), _heads(k, b, s, heads), _heads(v, b, s, heads),
                                       dropout_p=dropout, is_causal=causal)
    a = F.linear(nb.reshape(nb.swap_axes(a, 1, 2), (b, s, d)), p["wo"], p["bo"])
    x = x + F.dropout(a, dropout)
    h = F.layer_norm(x, p["ln2_w"], p["ln2_b"])
    h = F.linear(nb.gelu(F.linear(h, p["w1"], p["b1"])), p["w2"], p["b2"])
    return x + F.dropout(h, dropout)


@functools.lru_cache(maxsize=None)
def _block_program(heads: int, causal: bool, dropout: float, optimizer: bool):
    def loss_fn(params, x):
        out = _block(x, params, heads, causal, dropout)
        return nb.mean(out * out)

    if not optimizer:
        return nb.compile(lambda params, x: nb.value_and_grad(loss_fn)(params, x))

    def step(params, opt, x):
        loss, grads = nb.value_and_grad(loss_fn)(params, x)
        return loss, *_adamw(params, grads, opt)

    return nb.compile(step)


def _decoder(base, ids, heads, adapters=None):
    x = F.embedding(ids, base["embed"])
    for i, layer in enumerate(base["layers"]):
        x = _block(x, layer, heads, True, lora=adapters[i] if adapters is not None else None)
    return F.layer_norm(x, base["lnf_w"], base["lnf_b"]) @ base["head"]


@functools.lru_cache(maxsize=None)
def _decoder_program(heads: int):
    return nb.compile(lambda base, ids: _decoder(base, ids, heads))


@functools.lru_cache(maxsize=None)
def _lora_program(heads: int):
    def loss_fn(adapters, base, ids):
        return F.cross_entropy_loss(_decoder(base, ids, heads, adapters), ids)

    return nb.compile(lambda adapters, base, ids: nb.value_and_grad(loss_fn)(adapters, base, ids))


def _cnn(p, img):
    h = nb.relu(nb.conv2d(img, p["k1"], padding=1, bias=p["b1"]))
    h = nb.relu(nb.conv2d(h, p["k2"], padding=1, bias=p["b2"]))
    h = nb.max_pool2d(h, kernel_size=2)
    h = nb.relu(nb.conv2d(h, p["k3"], padding=1, bias=p["b3"]))
    return F.linear(nb.mean(h, axis=(1, 2)), p["wl"], p["bl"])


@nb.compile
def _cnn_classify(p, img):
    logits = _cnn(p, img)
    return logits, nb.argmax(logits, axis=-1)


@nb.compile
def _cnn_step(p, img, labels):
    return nb.value_and_grad(lambda p, img, labels: F.cross_entropy_loss(_cnn(p, img), labels))(p, img, labels)


@functools.lru_cache(maxsize=None)
def _qlora_program(width: int, ff: int):
    def weight(codes, shape):
        n = shape[0] * shape[1]
        return dict(codes, original_shape=shape, original_numel=n, padded_numel=n, block_size=64)

    def loss_fn(adapters, up, down, x):
        lin = functools.partial(nb.nn.finetune.qlora_linear, alpha=16.0, compute_dtype=nb.DType.bfloat16)
        h = nb.gelu(lin(x, weight(up, (width, ff)), adapters["up"]))
        out = x + lin(h, weight(down, (ff, width)), adapters["down"])
        return nb.mean(out * out)

    return nb.compile(lambda adapters, up, down, x: nb.value_and_grad(loss_fn)(adapters, up, down, x))


# ---- what a program has in hand -------------------------------------------------------------------
class _Maker:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int, dtype: str = "float32"):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = getattr(torch, dtype)

    def __call__(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.gen, device="cuda")
        return nb.Tensor.from_dlpack(t.mul_(std).add_(mean).to(self.dtype))

    def uniform(self, *shape):
        return nb.Tensor.from_dlpack(torch.rand(shape, generator=self.gen, device="cuda").to(self.dtype))

    def ints(self, hi, *shape):
        return nb.Tensor.from_dlpack(torch.randint(0, hi, shape, generator=self.gen, device="cuda"))

    def block(self, d, ff, layers=1):
        w = d ** -0.5
        # (queries and keys of a trained layer: scores of a standard deviation of about 2; what a
        # block adds to the stream falls with the number of blocks)
        out = (2.0 * layers) ** -0.5
        p = {"wq": self(d, d, std=1.4 * w), "wk": self(d, d, std=1.4 * w), "wv": self(d, d, std=w),
             "wo": self(d, d, std=out * w), "w1": self(d, ff, std=w), "w2": self(ff, d, std=out * ff ** -0.5)}
        p.update({n: self(1, d, std=0.1) for n in ("bq", "bv", "bo", "b2")}, b1=self(1, ff, std=0.1))
        p.update({n: self(d, std=0.1, mean=1.0) for n in ("ln1_w", "ln2_w")})
        p.update({n: self(d, std=0.1) for n in ("ln1_b", "ln2_b")})
        return p

    def decoder(self, case):
        d, v = case["width"], case["vocab"]
        return {"embed": self(v, d), "head": self(d, v, std=d ** -0.5), "lnf_w": self(d, std=0.1, mean=1.0),
                "lnf_b": self(d, std=0.1), "layers": [self.block(d, case["ff"], case["layers"]) for _ in range(case["layers"])]}

    def adapter(self, d_in, d_out, rank):
        return {"A": self(d_in, rank, std=d_in ** -0.5), "B": self(rank, d_out, std=0.02)}

    def moments(self, params, small):
        """AdamW's state after some steps: moments of gradients of about the size ``small``."""
        leaves, tree = nb.tree_flatten(params)
        m = [self(*t.shape, std=small) for t in leaves]
        v = [nb.Tensor.from_dlpack((torch.rand(tuple(t.shape), generator=self.gen, device="cuda") + 0.5)
                                   .mul_(small * small).to(self.dtype)) for t in leaves]
        return {"m": nb.tree_unflatten(tree, m), "v": nb.tree_unflatten(tree, v),
                "step": nb.Tensor.from_dlpack(torch.full((), 10.0, device="cuda"))}

    def codes(self, rows, cols):
        """A weight as four-bit codes with a scale per block of 64 (the format of ``quantize_nf4``)."""
        w = torch.randn((rows * cols // 64, 64), generator=self.gen, device="cuda").mul_(rows ** -0.5)
        scale = w.abs().amax(dim=1)
        level = torch.from_numpy(NF4_LEVELS).to("cuda")
        idx = torch.bucketize((w / scale[:, None]).reshape(-1), (level[1:] + level[:-1]) / 2).to(torch.uint8)
        return {"indices": nb.Tensor.from_dlpack(idx), "scales": nb.Tensor.from_dlpack(scale)}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "mlp":
        mk = _Maker(seed)
        sizes = [case["width_in"]] + [case["hidden"]] * case["depth"] + [case["width_out"]]
        params = [(mk(a, b, std=(2.0 / a) ** 0.5), mk(1, b, std=0.1)) for a, b in zip(sizes, sizes[1:])]
        args = [params, mk(case["batch"], sizes[0]), mk(case["batch"], sizes[-1])]
        step = _mlp_step
        if case["optimizer"]:
            step = _mlp_update
            args.insert(1, mk.moments(params, 0.05))
        return dict(step=_compiled(step) if case["compiled"] else step, args=args, eager=not case["compiled"])
    if kind == "chain":
        mk = _Maker(seed, case["dtype"])
        return dict(step=_chain_step, args=[mk(case["rows"], case["cols"]) for _ in range(2)])
    if kind == "rows":
        mk = _Maker(seed, case["dtype"])
        shape = (case["rows"], case["cols"])
        return dict(step=_rows_step, args=[mk(*shape), mk(*shape), mk(shape[1], std=0.1, mean=1.0),
                                           mk(shape[1], std=0.1), mk.uniform(*shape)])
    if kind == "block":
        mk = _Maker(seed, case["dtype"])
        if case["dropout"]:
            nb.set_seed(seed)
        params = mk.block(case["width"], case["ff"])
        args = [params, mk(case["batch"], case["seq"], case["width"])]
        if case["optimizer"]:
            args.insert(1, mk.moments(params, 1e-3))
        return dict(step=_block_program(case["heads"], case["causal"], case["dropout"], case["optimizer"]), args=args)
    if kind == "cnn":
        mk = _Maker(seed)
        c0, c1, c2, c3 = (case[c] for c in ("c0", "c1", "c2", "c3"))
        p = {"k%d" % (i + 1): mk(3, 3, a, b, std=(2.0 / (9 * a)) ** 0.5)
             for i, (a, b) in enumerate(((c0, c1), (c1, c2), (c2, c3)))}
        p.update({"b%d" % (i + 1): mk(c, std=0.1) for i, c in enumerate((c1, c2, c3))})
        p.update(wl=mk(c3, case["classes"], std=(2.0 / c3) ** 0.5), bl=mk(1, case["classes"], std=0.1))
        img = mk.uniform(case["batch"], case["hw"], case["hw"], c0)
        if not case["train"]:
            return dict(step=_cnn_classify, args=[p, img])
        return dict(step=_cnn_step, args=[p, img, mk.ints(case["classes"], case["batch"])])
    if kind in ("decoder", "lora"):
        mk = _Maker(seed, "bfloat16")
        base, ids = mk.decoder(case), mk.ints(case["vocab"], case["batch"], case["seq"])
        if kind == "decoder":
            return dict(step=_decoder_program(case["heads"]), args=[base, ids])
        d, r = case["width"], case["rank"]
        adapters = [{"q": mk.adapter(d, d, r), "v": mk.adapter(d, d, r)} for _ in range(case["layers"])]
        return dict(step=_lora_program(case["heads"]), args=[adapters, base, ids])
    if kind == "qlora":
        mk = _Maker(seed, "bfloat16")
        d, ff, r = case["width"], case["ff"], case["rank"]
        return dict(step=_qlora_program(d, ff),
                    args=[{"up": mk.adapter(d, ff, r), "down": mk.adapter(ff, d, r)}, mk.codes(d, ff),
                          mk.codes(ff, d), mk(case["tokens"], d)])
    raise ValueError(kind)


_compiled = functools.lru_cache(maxsize=None)(nb.compile)


def run(state: dict):
    out = state["step"](*state["args"])
    if state.get("eager"):
        nb.realize_all(*nb.tree_leaves(out))
    return nb.tree_map(lambda t: t.to_torch(), out)


# ---- what a pass cannot do without ---------------------------------------------------------------
def _block_work(case, tokens, train, frozen=False):
    """(weights, flops) of one block; attention counts the visible half of causal scores."""
    d, ff = case["width"], case["ff"]
    weights = 4 * d * d + 2 * d * ff
    products = 2 * tokens * weights
    scores = 4 * tokens * case["seq"] * d * (0.5 if case.get("causal", True) else 1.0)
    if not train:
        return weights, products + scores
    return weights, products * (2 if frozen else 3) + 3.5 * scores


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "mlp":
        sizes = [case["width_in"]] + [case["hidden"]] * case["depth"] + [case["width_out"]]
        n = sum(a * b + b for a, b in zip(sizes, sizes[1:]))
        pair = [2 * case["batch"] * a * b for a, b in zip(sizes, sizes[1:])]
        moved = n * (6 if case["optimizer"] else 2) + case["batch"] * (sizes[0] + sizes[-1])
        return {"bytes": 4 * moved, "flops": 3 * sum(pair) - pair[0]}
    if kind in ("chain", "rows"):
        size = 4 if case["dtype"] == "float32" else 2
        n = case["rows"] * case["cols"]
        return {"bytes": size * n * (3 if kind == "chain" else 5), "flops": n * (12 if kind == "chain" else 40)}
    if kind == "block":
        size = 4 if case["dtype"] == "float32" else 2
        tokens = case["batch"] * case["seq"]
        weights, flops = _block_work(case, tokens, True)
        flops -= 6 * tokens * case["width"] ** 2  # (no gradient of the block's input is asked for)
        moved = weights * (6 if case["optimizer"] else 2) + tokens * case["width"]
        return {"bytes": size * moved, "flops": flops}
    if kind in ("decoder", "lora"):
        tokens, d, v = case["batch"] * case["seq"], case["width"], case["vocab"]
        weights, flops = _block_work(case, tokens, kind == "lora", frozen=True)
        head = 2 * tokens * d * v
        moved = case["layers"] * weights + d * v + tokens * d
        if kind == "decoder":
            return {"bytes": 2 * (moved + tokens * v), "flops": case["layers"] * flops + head}
        adapters = 12 * tokens * 4 * d * case["rank"] * case["layers"]
        return {"bytes": 2 * moved, "flops": case["layers"] * flops + 2 * head + adapters}
    if kind == "cnn":
        n, hw = case["batch"] * case["hw"] ** 2, case["hw"]
        c = [case[k] for k in ("c0", "c1", "c2", "c3")]
        pair = [18 * n * c[0] * c[1], 18 * n * c[1] * c[2], 18 * (n // 4) * c[2] * c[3]]
        weights = 9 * (c[0] * c[1] + c[1] * c[2] + c[2] * c[3]) + c[3] * case["classes"]
        flops = 3 * sum(pair) - pair[0] if case["train"] else sum(pair)
        return {"bytes": 4 * (n * c[0] + weights * (2 if case["train"] else 1)), "flops": flops}
    t, d, ff, r = case["tokens"], case["width"], case["ff"], case["rank"]
    return {"bytes": 2 * d * ff * (1 + 4 / 64) + 2 * t * d + 8 * r * (d + ff),
            "flops": 2 * t * d * ff * 3 + 12 * t * r * (d + ff)}


def tolerance(case: dict):
    """About four times the largest relative error of an output against the same step with wider
    numbers: float32 against double precision, bfloat16 against float32."""
    kind = case["kind"]
    if kind in ("decoder", "lora", "qlora") or kind == "block" and case["dtype"] == "bfloat16":
        return {"rel": 0.03}  # (bfloat16: 0.5 to 2.5e-2 after one to twelve layers)
    if case.get("dtype") == "bfloat16":
        return {"rel": 0.016}  # (one rounding of every input and result: 4e-3)
    # A unit whose input is zero to within rounding, or two maxima of one pooling window that are
    # as close, may fall on either side, and its part of a gradient with them.
    if kind == "mlp":
        return {"rel": 1.5e-3 if case["depth"] > 1 else 1e-4}  # (3e-4; one hidden layer: 5e-6, and rarely a unit)
    if kind == "cnn" and case["train"]:
        return {"rel": 1.6e-4}  # (4e-5)
    return {"rel": 2e-5, "max": 2e-3, "differ": 0.001}  # (sums 1e-7 to 4e-7, moments squared; class ids exact but for ties)
