"""The work this package does for its users, as cases that can be timed.

A case is one layer's training step (forward, then backward with every gradient) as one rank runs it: the
halo-exchange convolution, ring attention, the sharded LayerNorm, the spatially sharded GroupNorm, the
projections around attention and the Swin block. What travels between ranks is made from the seed and held
locally, so a case needs one GPU. ``listed`` names the cases, ``draw`` gives others of the same ranges.
"""

from __future__ import annotations

import itertools
import math

import torch

from jigsaw_amd import attention, groupnorm, layernorm, projection, swin
from jigsaw_amd.conv import HipConvNdConfig, TileGroup, _ConvNd
from jigsaw_amd.halo import HaloGeometry

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

# Nothing drawn goes beyond the listed cases: the convolution of configuration 2 and the ring of configuration 4.
# fp32 has a sixteenth of the matrix rate, a strided layer does the same arithmetic on four times the cells.
_MOST_CONV_FLOPS = 3 * 2 * 8 * 64 * 64 * 9 * 1024 * 1024
_MOST_RING_FLOPS = 14 * 8 * 4096 * 4 * 4096 * 64


def listed() -> list:
    return [
        # The example model's first layer (fp32, RGB images, a 256 x 256 tile of 512 x 512): launches and host time count.
        {"name": "conv2d_example", "op": "conv", "dtype": "fp32", "batch": 4, "c_in": 3, "c_out": 16, "size": "256x256", "stride": 1, "mesh": 2},
        # The benchmark's layer: a 1024 x 1024 tile between eight neighbours, 64 channels.
        {"name": "conv2d_tile", "op": "conv", "dtype": "bf16", "batch": 8, "c_in": 64, "c_out": 64, "size": "1024x1024", "stride": 1, "mesh": 3},
        # A tile and channel counts that divide by nothing a kernel would like.
        {"name": "conv2d_ragged", "op": "conv", "dtype": "bf16", "batch": 2, "c_in": 40, "c_out": 72, "size": "217x301", "stride": 1, "mesh": 3},
        # The down-sampling layer between two stages of an encoder.
        {"name": "conv2d_down", "op": "conv", "dtype": "bf16", "batch": 4, "c_in": 64, "c_out": 128, "size": "256x256", "stride": 2, "mesh": 3},
        # A volume: 128^3 of 256^3, 26 neighbours.
        {"name": "conv3d_tile", "op": "conv", "dtype": "bf16", "batch": 2, "c_in": 32, "c_out": 32, "size": "128x128x128", "stride": 1, "mesh": 3},
        # Ring attention on a short sequence: latency.
        {"name": "ring_small", "op": "ring", "dtype": "bf16", "batch": 1, "heads": 4, "tokens": 128, "head_size": 32, "chunks": 2},
        # ViT ring attention, 16384 tokens on four ranks, half of the heads.
        {"name": "ring_vit", "op": "ring", "dtype": "bf16", "batch": 1, "heads": 8, "tokens": 4096, "head_size": 64, "chunks": 4},
        # A token count per rank that is no multiple of a tile.
        {"name": "ring_ragged", "op": "ring", "dtype": "bf16", "batch": 2, "heads": 12, "tokens": 1000, "head_size": 64, "chunks": 2},
        # The LayerNorm beside it: 512 channels over two ranks.
        {"name": "layernorm_vit", "op": "layernorm", "dtype": "bf16", "rows": 4096, "cols": 256},
        # GroupNorm behind the convolution of the benchmark.
        {"name": "groupnorm_tile", "op": "groupnorm", "dtype": "bf16", "batch": 8, "channels": 64, "groups": 8, "size": "1024x1024"},
        # The projections before and behind the attention core, 8 x 4096 tokens.
        {"name": "projections_vit", "op": "projections", "dtype": "bf16", "batch": 8, "tokens": 4096, "dim": 512, "heads": 8},
        # A Swin block on a 256 x 256-token tile, shifted windows.
        {"name": "swin_tile", "op": "swin", "dtype": "bf16", "batch": 1, "size": "256x256", "dim": 128, "shift": 4},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    op = rng.choice(("conv2d", "conv2d", "conv_down", "conv3d", "ring", "ring", "layernorm", "groupnorm", "projections", "swin"))
    while True:
        case = _DRAW[op](rng)
        most = _MOST_RING_FLOPS if case["op"] == "ring" else _MOST_CONV_FLOPS
        if work(case)["flops"] * (16 if case["dtype"] == "fp32" else 1) * case.get("stride", 1) ** 2 <= most:
            return case


def _draw_conv2d(rng) -> dict:
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
    most = 512 if dtype == "fp32" else 1024
    return {"op": "conv", "dtype": dtype, "batch": rng.randint(1, 8), "c_in": _log(rng, 3, 128), "c_out": _log(rng, 3, 128),
            "size": f"{_log(rng, 32, most)}x{_log(rng, 32, most)}", "stride": 1, "mesh": rng.choice((2, 3))}


def _draw_conv_down(rng) -> dict:
    return {"op": "conv", "dtype": "bf16", "batch": rng.randint(1, 8), "c_in": _log(rng, 16, 128), "c_out": _log(rng, 16, 256),
            "size": f"{2 * _log(rng, 16, 256)}x{2 * _log(rng, 16, 256)}", "stride": 2, "mesh": rng.choice((2, 3))}


def _draw_conv3d(rng) -> dict:
    size = "x".join(str(_log(rng, 12, 128)) for _ in range(3))
    return {"op": "conv", "dtype": "bf16", "batch": rng.randint(1, 2), "c_in": _log(rng, 4, 64), "c_out": _log(rng, 4, 64),
            "size": size, "stride": 1, "mesh": rng.choice((2, 3))}


def _draw_ring(rng) -> dict:
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
    tokens = _log(rng, 64, 1024 if dtype == "fp32" else 4096)
    return {"op": "ring", "dtype": dtype, "batch": rng.randint(1, 4), "heads": rng.randint(1, 16), "tokens": tokens,
            "head_size": rng.choice((32, 64, 64, 80, 96, 128)), "chunks": rng.randint(1, 8)}


def _draw_layernorm(rng) -> dict:
    cols = 4 * _log(rng, 16, 512)
    return {"op": "layernorm", "dtype": rng.choice(("bf16", "bf16", "fp32")), "rows": _log(rng, 256, min(1 << 18, (1 << 26) // cols)), "cols": cols}


def _draw_groupnorm(rng) -> dict:
    groups = rng.choice((4, 8, 16, 32))
    return {"op": "groupnorm", "dtype": rng.choice(("bf16", "bf16", "fp32")), "batch": rng.randint(1, 8), "channels": groups * rng.randint(1, 4),
            "groups": groups, "size": f"{_log(rng, 16, 512)}x{_log(rng, 16, 512)}"}


def _draw_projections(rng) -> dict:
    heads = rng.randint(2, 16)
    return {"op": "projections", "dtype": "bf16", "batch": rng.randint(1, 8), "tokens": _log(rng, 64, 4096), "dim": 64 * heads, "heads": heads}


def _draw_swin(rng) -> dict:
    return {"op": "swin", "dtype": "bf16", "batch": rng.randint(1, 4), "size": f"{8 * _log(rng, 4, 32)}x{8 * _log(rng, 4, 32)}",
            "dim": 32 * rng.randint(2, 8), "shift": rng.choice((0, 4))}


_DRAW = {"conv2d": _draw_conv2d, "conv_down": _draw_conv_down, "conv3d": _draw_conv3d, "ring": _draw_ring, "layernorm": _draw_layernorm,
         "groupnorm": _draw_groupnorm, "projections": _draw_projections, "swin": _draw_swin}


def _size(case) -> tuple:
    return tuple(int(v) for v in case["size"].split("x"))


# --------------------------------------------------------------------------- #
# what a user's program has in hand before the step
# --------------------------------------------------------------------------- #
def prepare(case: dict, seed: int) -> dict:
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)

    def normal(*shape, dtype=_DTYPES[case["dtype"]], std=1.0, mean=0.0):
        return torch.randn(*shape, device=device, generator=gen).mul_(std).add_(mean).to(dtype)

    state = _PREPARE[case["op"]](case, normal, device)
    state["op"] = case["op"]
    return state


class _HeldStrips:
    """The halo exchange of one rank whose neighbours' strips are already here; keeps what the rank sends."""

    def __init__(self, forward: dict, backward: dict) -> None:
        self._forward, self._backward = forward, backward
        self.sent: dict = {}

    def forward(self, send: dict) -> dict:
        self.sent["forward"] = send
        return self._forward

    def backward(self, send: dict) -> dict:
        self.sent["backward"] = send
        return self._backward


def _prepare_conv(case, normal, device) -> dict:
    size, n = _size(case), len(_size(case))
    kernel, stride, padding, dilation = (3,) * n, (case["stride"],) * n, (1,) * n, (1,) * n
    # mesh 3: a rank between neighbours on every side; mesh 2: a corner of the domain
    rank = 1 if case["mesh"] == 3 else 0
    groups = tuple(TileGroup(case["mesh"], rank) for _ in size)
    geom = HaloGeometry.for_conv(size, kernel, stride, padding, dilation, (rank,) * n, (case["mesh"],) * n)
    lead_x = (case["batch"], case["c_in"])
    present = [o for o in itertools.product((-1, 0, 1), repeat=n) if any(o) and all(0 <= rank + v < case["mesh"] for v in o)]
    exchange = _HeldStrips({o: normal(*lead_x, *geom.strip_extent(o, "assemble")) for o in present},
                           {o: normal(*lead_x, *geom.strip_extent(o, "fold")) for o in present})
    bound = 1.0 / math.sqrt(case["c_in"] * 3**n)
    w = normal(case["c_out"], case["c_in"], *kernel, std=bound).requires_grad_()
    b = normal(case["c_out"], std=bound).requires_grad_()
    out = tuple(s // case["stride"] for s in size)
    return {
        "x": normal(*lead_x, *size).requires_grad_(), "w": w, "b": b, "grad": normal(case["batch"], case["c_out"], *out),
        "args": (stride, padding, dilation, groups, None), "exchange": exchange,
        "config": HipConvNdConfig.for_rank(n, b, exchange),
    }


def _prepare_ring(case, normal, device) -> dict:
    d = case["head_size"]
    shape = (case["batch"], case["heads"], case["tokens"], d)
    chunk = lambda: normal(*shape, std=d**-0.5)  # noqa: E731
    return {"q": chunk(), "k": [chunk() for _ in range(case["chunks"])], "v": [chunk() for _ in range(case["chunks"])],
            "grad": normal(*shape), "scale": d**-0.5}


class _OtherShard:
    """A channel group of two whose other rank's contributions are already here, in the order they are asked for."""

    def __init__(self, contributions: list) -> None:
        self._contributions, self._turn = contributions, 0

    def size(self) -> int:
        return 2

    def all_reduce(self, t: torch.Tensor, op: str) -> None:
        other = self._contributions[self._turn % len(self._contributions)]
        self._turn += 1
        if op == "avg":
            t.lerp_(other.view_as(t), 0.5)
        else:
            t.add_(other.view_as(t))


def _prepare_layernorm(case, normal, device) -> dict:
    rows, cols = case["rows"], case["cols"]
    f32 = torch.float32
    group = _OtherShard([
        normal(rows, dtype=f32, std=cols**-0.5),              # the other half's mean
        normal(rows, dtype=f32, std=0.05, mean=1.0).abs_(),   # its variance about the common mean
        normal(rows, dtype=f32, std=cols**-0.5),              # backward: its mean of g * weight
        normal(rows, dtype=f32, std=cols**0.5),               # and its sum of g * weight * x_hat
    ])
    return {"x": normal(rows, cols).requires_grad_(), "w": normal(cols, std=0.2, mean=1.0).requires_grad_(),
            "b": normal(cols, std=0.2).requires_grad_(), "grad": normal(rows, cols), "group": group}


def _prepare_groupnorm(case, normal, device) -> dict:
    c, shape = case["channels"], (case["batch"], case["channels"], *_size(case))
    return {"x": normal(*shape).requires_grad_(), "w": normal(c, std=0.2, mean=1.0).requires_grad_(),
            "b": normal(c, std=0.2).requires_grad_(), "grad": normal(*shape), "groups": case["groups"]}


def _prepare_projections(case, normal, device) -> dict:
    b, s, c, h = case["batch"], case["tokens"], case["dim"], case["heads"]
    return {
        "x": normal(b, s, c).requires_grad_(), "heads_out": normal(b, h, s, c // h).requires_grad_(), "heads": h,
        "qkv_w": normal(3 * c, c, std=c**-0.5).requires_grad_(), "qkv_b": normal(3 * c, std=0.1).requires_grad_(),
        "out_w": normal(c, c, std=c**-0.5).requires_grad_(), "out_b": normal(c, std=0.1).requires_grad_(),
        "qkv_grad": normal(3, b, h, s, c // h), "out_grad": normal(b, s, c),
    }


def _prepare_swin(case, normal, device) -> dict:
    tile, dim = _size(case), case["dim"]
    # heads of 32 channels in 8 x 8 windows; fp32 parameters, the tokens in bf16 under autocast
    block = swin.SwinBlock(dim, dim // 32, 8, tile, shift=case["shift"], device=device)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if "norm" in name and name.endswith("weight"):
                p.copy_(normal(*p.shape, dtype=p.dtype, std=0.1, mean=1.0))
            else:
                p.copy_(normal(*p.shape, dtype=p.dtype, std=p.shape[1] ** -0.5 if p.dim() == 2 and "bias_table" not in name else 0.1))
    shape = (case["batch"], *tile, dim)
    return {"block": block, "params": list(block.parameters()), "x": normal(*shape).requires_grad_(), "grad": normal(*shape)}


_PREPARE = {"conv": _prepare_conv, "ring": _prepare_ring, "layernorm": _prepare_layernorm, "groupnorm": _prepare_groupnorm,
            "projections": _prepare_projections, "swin": _prepare_swin}


# --------------------------------------------------------------------------- #
# one step
# --------------------------------------------------------------------------- #
def run(state: dict):
    return _RUN[state["op"]](state)


def _run_conv(s):
    y = _ConvNd.apply(s["x"], s["w"], s["b"], *s["args"], s["config"])[0]
    grads = torch.autograd.grad(y, (s["x"], s["w"], s["b"]), s["grad"])
    sent = s["exchange"].sent
    return [y, *grads, *sent["forward"].values(), *sent["backward"].values()]


def _run_ring(s):
    out, lse = attention.ring_forward(s["q"], s["k"], s["v"], s["scale"])
    dq, dk, dv = attention.ring_backward(s["grad"], s["q"], out, lse, s["k"], s["v"], s["scale"])
    return [out, lse, dq, *dk, *dv]


def _run_layernorm(s):
    y = layernorm.layer_norm(s["x"], s["w"], s["b"], s["group"])
    return [y, *torch.autograd.grad(y, (s["x"], s["w"], s["b"]), s["grad"])]


def _run_groupnorm(s):
    y = groupnorm.group_norm(s["x"], s["groups"], s["w"], s["b"])
    return [y, *torch.autograd.grad(y, (s["x"], s["w"], s["b"]), s["grad"])]


def _run_projections(s):
    qkv = projection.qkv_projection(s["x"], s["qkv_w"], s["qkv_b"], s["heads"])
    y = projection.heads_projection(s["heads_out"], s["out_w"], s["out_b"])
    into = (s["x"], s["qkv_w"], s["qkv_b"], s["heads_out"], s["out_w"], s["out_b"])
    return [qkv, y, *torch.autograd.grad((qkv, y), into, (s["qkv_grad"], s["out_grad"]))]


def _run_swin(s):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = s["block"](s["x"])
    return [y, *torch.autograd.grad(y, (s["x"], *s["params"]), s["grad"])]


_RUN = {"conv": _run_conv, "ring": _run_ring, "layernorm": _run_layernorm, "groupnorm": _run_groupnorm,
        "projections": _run_projections, "swin": _run_swin}


# --------------------------------------------------------------------------- #
# what a step cannot do without, and how close two right answers are
# --------------------------------------------------------------------------- #
def work(case: dict) -> dict:
    op, es = case["op"], _BYTES[case["dtype"]]
    if op == "conv":
        size = _size(case)
        cells, out = math.prod(size), math.prod(s // case["stride"] for s in size)
        taps = 3 ** len(size)
        weights = case["c_in"] * case["c_out"] * taps
        # x and gx, y and its gradient, the weights and theirs; the strips are small beside them
        return {"bytes": es * (2 * case["batch"] * (case["c_in"] * cells + case["c_out"] * out) + 2 * weights),
                "flops": 3 * 2 * case["batch"] * weights * out}
    if op == "ring":
        rows = case["batch"] * case["heads"] * case["tokens"]
        # q, out, dq and the output gradient; k, v and their gradients per chunk
        return {"bytes": rows * case["head_size"] * es * (4 + 4 * case["chunks"]),
                "flops": 14 * rows * case["tokens"] * case["chunks"] * case["head_size"]}
    if op == "layernorm":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n * es, "flops": 20 * n}
    if op == "groupnorm":
        n = case["batch"] * case["channels"] * math.prod(_size(case))
        return {"bytes": 4 * n * es, "flops": 20 * n}
    if op == "projections":
        rows, c = case["batch"] * case["tokens"], case["dim"]
        # x, its gradient, qkv and its gradient (three times as wide); the same for the output projection
        return {"bytes": es * (rows * c * (2 + 6 + 4) + 8 * c * c), "flops": 3 * 2 * rows * c * 4 * c}
    # the Swin block: qkv, output projection and MLP are 12 dim^2 weights; attention sees 64 keys a token
    tokens, c = case["batch"] * math.prod(_size(case)), case["dim"]
    return {"bytes": 4 * tokens * c * es + 2 * 12 * c * c * 4, "flops": tokens * (3 * 2 * 12 * c * c + 14 * 64 * c)}


def tolerance(case: dict) -> dict:
    # fp32 sums in another order; one rounding to 16 bits here and there (weights and tokens pass through several in a block)
    return {"rel": {"fp32": 1e-5, "fp16": 3e-3, "bf16": 1e-2}[case["dtype"]]}
