"""The work this library is called for, as cases that can be timed and checked one by one.

A case is one of four kinds of call:

- `linear`: one encoded leaf's forward on a 16-bit activation, called eagerly, as a diffusion
  transformer's layers are called over its image and text tokens;
- `step`: the four linears of one transformer block (QKV, attention output, MLP up and down) at a
  few rows, captured into a HIP graph and replayed, as a decode loop runs them: each linear reads
  the activation that attention or the MLP's activation function would hand it;
- `modulated`: `int8_rows` (layer norm, the block's scale and shift tables, rotation and
  quantization in one pass) and the int8 leaf that reads its rows, as a DiT block's first half runs;
- `bake`: a LoRA baked into a copy of a stored weight, as a request that brings one does.

The widths are those of the benchmark (`bench.py`): 3072-wide DiT blocks with a 12288-wide MLP, and
4096-wide language blocks with a 14336-wide one. Weights and activations are drawn on the GPU from
the seed; activations are N(0, 1) with 1% of their channels twenty times larger, which is what
per-token quantization and the rotation are there for.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "cozy-runtime_amd"))

from cozyq import bake, leaves, operands  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
E4M3 = torch.float8_e4m3fn
#: The largest products a case may take, in multiply-adds: one 4096-row pass through a 3072 x 12288
#: layer; the W4A4 formats, which do more work an element, a quarter of it.
MOST_MACS = 4096 * 3072 * 12288
#: The 16-level codebook of w4a8.convrot weights: a Lloyd-Max fit of a normal distribution.
CODEBOOK = (
    -0.980602, -0.794529, -0.638165, -0.500986, -0.377321, -0.263187, -0.155210, -0.050720,
    0.052541, 0.156985, 0.265284, 0.379533, 0.502636, 0.638953, 0.794876, 0.980671,
)  # fmt: skip
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _case(kind: str, fmt: str, rows: int, k: int, n: int, dtype: str = "bf16", bias: bool = True,
          rank: int = 0) -> dict:  # fmt: skip
    return {"kind": kind, "format": fmt, "rows": rows, "k": k, "n": n, "dtype": dtype, "bias": bias,
            "rank": rank}  # fmt: skip


def listed() -> list[dict]:
    return [
        # One token through one small layer, called eagerly: what a call costs when there is
        # hardly any work in it.
        dict(_case("linear", "int8", 1, 3072, 3072), name="int8_one_row"),
        # The DiT's MLP up-projection over 4096 image tokens, the library's headline shape.
        dict(_case("linear", "int8", 4096, 3072, 12288), name="int8_ffn_up_4096"),
        # A modulated block's norm, tables and QKV on an image and its text, an odd number of rows.
        dict(_case("modulated", "int8", 1179, 3072, 9216), name="int8_modulated_qkv_1179"),
        # One language block's linears for one token.
        dict(_case("step", "fp8", 1, 4096, 14336, bias=False), name="fp8_step_1"),
        # A short prompt through a language block's MLP up-projection.
        dict(_case("linear", "fp8", 300, 4096, 14336, bias=False), name="fp8_ffn_up_300"),
        # The same layer over a whole 4096-token prompt.
        dict(_case("linear", "fp8", 4096, 4096, 14336, bias=False), name="fp8_ffn_up_4096"),
        # The DiT's MLP down-projection in MX blocks: a long reduction, few columns.
        dict(_case("linear", "mxfp8", 4096, 12288, 3072), name="mxfp8_ffn_down_4096"),
        # Sixteen sequences' decode step on 4-bit weights with int8 activations.
        dict(_case("step", "w4a8", 16, 3072, 12288), name="w4a8_step_16"),
        # Five sequences' decode step on nvfp4 weights with fp16 activations.
        dict(_case("step", "nvfp4", 5, 4096, 14336, dtype="fp16", bias=False), name="nvfp4_step_5"),
        # W4A4 with its low-rank branch: the DiT's square layer over 4096 tokens, int4 groups.
        dict(_case("linear", "svdq_int4", 4096, 3072, 3072, rank=32), name="svdq_int4_4096"),
        # W4A4 in nvfp4 blocks: QKV over an odd number of tokens.
        dict(_case("linear", "svdq_nvfp4", 1531, 3072, 9216, rank=32), name="svdq_nvfp4_qkv_1531"),
        # A request's rank-32 LoRA baked into an int8.convrot MLP weight.
        dict(_case("bake", "int8", 12288, 3072, 32), name="bake_int8_12288"),
    ]


def _log(rng, low: float, high: float) -> float:
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng) -> dict:
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    bias = rng.random() < 0.5
    kind = rng.choice(("linear",) * 7 + ("step",) * 4 + ("modulated", "bake"))
    if kind == "step":
        fmt = rng.choice(("int8", "fp8", "w4a8", "nvfp4"))
        k = 256 * rng.randint(4, 16)
        n = 256 * rng.randint(2 * (k // 256), min(4 * (k // 256), 56))
        return _case(kind, fmt, round(_log(rng, 1, 64)), k, n, dtype, bias)
    if kind == "bake":
        fmt = rng.choice(("int8", "bf16"))
        return _case(kind, fmt, 8 * round(_log(rng, 128, 1536)), 256 * rng.randint(4, 12),
                     rng.choice((4, 8, 16, 32, 64)))  # fmt: skip
    fmt = "int8"
    if kind == "linear":
        fmt = rng.choice(("int8", "int8", "fp8", "fp8", "mxfp8", "w4a8", "svdq_int4", "svdq_nvfp4"))
    svdq = fmt.startswith("svdq")
    k = 256 * round(_log(rng, 4, 48 if kind == "linear" and not svdq else 16))
    n = 8 * round(_log(rng, 128, 1792))
    most = MOST_MACS // 4 if svdq else MOST_MACS
    few = kind == "linear" and not svdq and rng.random() < 0.25  # eager calls of a few rows
    rows = round(_log(rng, 1, 64) if few else _log(rng, 65, 4096))
    rows = max(1, min(rows, most // (k * n)))
    return _case(kind, fmt, rows, k, n, dtype, bias, rng.choice((32, 64)) if svdq else 0)


# ------------------------------------------------------------------------------ inputs


def _activations(rows: int, k: int, gen, dtype) -> torch.Tensor:
    x = torch.randn(rows, k, generator=gen, device="cuda")
    loud = torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 100)]
    x[:, loud] *= 20
    return x.to(dtype)


def _rowwise(w: torch.Tensor, most: float) -> tuple[torch.Tensor, torch.Tensor]:
    scale = (w.abs().amax(1) / most).clamp(min=1e-12)
    return w / scale[:, None], scale


def _nibbles(codes: torch.Tensor) -> torch.Tensor:
    """Codes 0..15 [N, K] packed two a byte, element 2k in the low nibble."""
    u = codes.to(torch.uint8)
    return (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()


def _nearest(v: torch.Tensor, levels: torch.Tensor) -> torch.Tensor:
    """The index of the level nearest to each value; `levels` ascending."""
    return torch.bucketize(v, (levels[1:] + levels[:-1]) / 2)


def _nvfp4_weight(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Packed E2M1 codes [N, K/2], E4M3 block scales [N, K/16] and the second level [1]."""
    n, k = w.shape
    second = (w.abs().amax() / (448 * 6)).reshape(1)
    blocks = w.view(n, k // 16, 16)
    scale = (blocks.abs().amax(-1) / (6 * second)).clamp(2.0**-9, 448).to(E4M3)
    ratio = blocks / (scale.float() * second)[..., None]
    codes = _nearest(ratio.abs(), torch.tensor(E2M1, device=w.device)) + 8 * (ratio < 0)
    return _nibbles(codes.view(n, k)), scale, second


def _weight(fmt: str, n: int, k: int, rank: int, gen) -> dict:
    """The stored parts of one weight, as a checkpoint of the format holds them."""
    w = torch.randn(n, k, generator=gen, device="cuda") * 0.02
    if fmt == "int8":
        q, scale = _rowwise(w, 127)
        return {"weight": q.round().to(torch.int8), "scale": scale}
    if fmt == "fp8":
        q, scale = _rowwise(w, 448)
        return {"weight": q.to(E4M3), "scale": scale}
    if fmt == "mxfp8":
        q, byte = _mx(w)
        return {"weight": q, "scale": byte}
    if fmt == "w4a8":
        q, scale = _rowwise(w, 127)
        book = torch.tensor(CODEBOOK, device="cuda")
        groups = q.view(n, k // 16, 16)
        group_scale = (groups.abs().amax(-1) / book.abs().amax()).to(E4M3)
        codes = _nearest(groups / group_scale.float().clamp(min=1e-6)[..., None], book)
        return {"weight": _nibbles(codes.view(n, k)), "group_scale": group_scale, "scale": scale,
                "codebook": book}  # fmt: skip
    if fmt == "nvfp4":
        weight, scale, second = _nvfp4_weight(w)
        return {"weight": weight, "scale": scale, "scale_2": second}
    smooth = torch.rand(k, generator=gen, device="cuda") * 1.5 + 0.5
    branch = {"pre_quant_scale": smooth,
              "lowrank_down": (torch.randn(rank, k, generator=gen, device="cuda") * 0.02).bfloat16(),
              "lowrank_up": (torch.randn(n, rank, generator=gen, device="cuda") * 0.02).bfloat16()}  # fmt: skip
    w = w / smooth
    if fmt == "svdq_int4":
        groups = w.view(n, k // 64, 64)
        scale = (groups.abs().amax(-1) / 7).half()
        codes = (groups / scale.float()[..., None]).round().clamp(-8, 7).to(torch.int8).view(n, k)
        return {"weight": _nibbles(codes & 15), "scale": scale, **branch}
    weight, scale, second = _nvfp4_weight(w)
    return {"weight": weight, "scale": scale, "scale_2": second, **branch}


_PROVIDERS = {
    "int8": lambda: leaves.Int8ConvRotNativeLeaf(),
    "fp8": lambda: leaves.RowwiseNativeLeaf(),
    "mxfp8": lambda: leaves.MicroScaledNativeLeaf(),
    "w4a8": lambda: leaves.W4a8NativeLeaf(),
    "nvfp4": lambda: leaves.Nvfp4NativeLeaf(),
    "svdq_int4": lambda: leaves.SvdqInt4NativeLeaf(),
    "svdq_nvfp4": lambda: leaves.SvdqNvfp4NativeLeaf(),
}


def _layers(case: dict) -> list[tuple[int, int]]:
    """The (inputs, outputs) of the case's linears."""
    k, n = case["k"], case["n"]
    return [(k, 3 * k), (k, k), (k, n), (n, k)] if case["kind"] == "step" else [(k, n)]


def _drawn(case: dict, seed: int) -> SimpleNamespace:
    """Everything the case draws from its seed: per linear its activation, stored parts and bias;
    the modulation tables; the LoRA's factors."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "bake":
        rows, k, rank = case["rows"], case["k"], case["n"]
        stored = torch.randn(rows, k, generator=gen, device="cuda") * 0.02
        if case["format"] == "int8":
            q, scale = _rowwise(stored, 127)
            parts = {"weight": q.round().to(torch.int8), "scale": scale}
        else:
            parts = {"value": stored.bfloat16()}
        down = (torch.randn(rank, k, generator=gen, device="cuda") * 0.02).bfloat16()
        up = (torch.randn(rows, rank, generator=gen, device="cuda") * 0.02).bfloat16()
        return SimpleNamespace(parts=parts, down=down, up=up, noise=seed & 0x7FFFFFFF)
    linears = []
    for k, n in _layers(case):
        x = _activations(case["rows"], k, gen, dtype)
        parts = _weight(case["format"], n, k, case["rank"], gen)
        bias = (torch.randn(n, generator=gen, device="cuda") * 0.1).to(dtype) if case["bias"] else None
        linears.append(SimpleNamespace(x=x, parts=parts, bias=bias))
    tables = None
    if case["kind"] == "modulated":
        tables = [(torch.randn(1, case["k"], generator=gen, device="cuda") * 0.2).to(dtype) for _ in range(2)]
    return SimpleNamespace(linears=linears, tables=tables)


def prepare(case: dict, seed: int) -> dict:
    drawn = _drawn(case, seed)
    if case["kind"] == "bake":
        baked = {role: t.clone() for role, t in drawn.parts.items()}
        return {"kind": "bake", "stored": drawn.parts, "baked": baked, "down": drawn.down, "up": drawn.up,
                "seed": drawn.noise}  # fmt: skip
    dtype = DTYPES[case["dtype"]]
    provider = _PROVIDERS[case["format"]]()
    built = [provider.leaf(torch, v.parts, SimpleNamespace(bias=v.bias), dtype) for v in drawn.linears]
    xs = [v.x for v in drawn.linears]
    state = {"kind": case["kind"], "leaves": built, "xs": xs, "tables": drawn.tables}
    if case["kind"] == "step":
        # A decode loop's step: warmed once on a side stream, then captured.
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.no_grad(), torch.cuda.stream(side):
            for leaf, x in zip(built, xs):
                leaf(x)
            side.synchronize()
            with torch.cuda.graph(graph, stream=side):
                outs = [leaf(x) for leaf, x in zip(built, xs)]
        torch.cuda.current_stream().wait_stream(side)
        state.update(graph=graph, outs=outs)
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["outs"]
    if kind == "bake":
        # The weight as stored replaces the last request's, then takes this one's LoRA.
        baked = state["baked"]
        for role in ("weight", "value"):
            if role in baked:
                baked[role].copy_(state["stored"][role])
        bake.bake(torch, baked, state["down"], state["up"], seed=state["seed"])
        return baked.get("weight", baked.get("value"))
    with torch.no_grad():
        (leaf,), (x,) = state["leaves"], state["xs"]
        if kind == "modulated":
            scale, shift = state["tables"]
            x = operands.int8_rows(x, (leaf,), norm="layer", eps=1e-6, scale=scale, shift=shift)
        return leaf(x)


# ------------------------------------------------------------------- work and tolerance

#: Stored bytes a weight, with its scales inside the row.
_WEIGHT_BYTES = {"int8": 1, "fp8": 1, "mxfp8": 1 + 1 / 32, "w4a8": 0.5 + 1 / 16, "nvfp4": 0.5 + 1 / 16,
                 "svdq_int4": 0.5 + 2 / 64, "svdq_nvfp4": 0.5 + 1 / 16}  # fmt: skip


def work(case: dict) -> dict:
    rows, rank = case["rows"], case["rank"]
    if case["kind"] == "bake":
        size = rows * case["k"] * (1 if case["format"] == "int8" else 2)
        factors = 2 * case["n"] * (rows + case["k"])
        return {"bytes": 2 * size + factors, "flops": 2 * rows * case["k"] * case["n"]}
    nbytes, flops = 0, 0
    for k, n in _layers(case):
        nbytes += 2 * rows * (k + n) + n * k * _WEIGHT_BYTES[case["format"]] + 4 * n
        nbytes += 2 * rank * (k + n) + (2 * n if case["bias"] else 0)
        flops += 2 * rows * k * n + 2 * rows * rank * (k + n)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    # int8 products are whole numbers and each rounding after them is the law's; a bake's noise is
    # its seed's.
    if case["kind"] == "bake" or (case["kind"] != "modulated" and case["format"] in ("int8", "w4a8")):
        return "exact"
    # float32 sums in another order, then one rounding to 16 bits, which moves to its neighbour for
    # some values; a norm's last bit moves some codes by one. Against 64 bits bf16 results are
    # 1.7e-3 off (2.4e-3 where the bias is added after a first rounding) and fp16 ones 2.1e-4 to
    # 3e-4: about four times that, less where the codes are whole.
    return {"rel": 1e-3 if case["dtype"] == "fp16" and case["kind"] != "modulated" else 7e-3}


# --------------------------------------------------------------- the same in 64 bits


def _over(v: torch.Tensor, by: float) -> torch.Tensor:
    """v / by, correctly rounded: torch multiplies by the reciprocal where `by` is a number."""
    return v / torch.full_like(v, by)


def _rotated(x: torch.Tensor) -> torch.Tensor:
    """x [M, K] float64 times the regular Hadamard matrix of 256 per 256 columns, orthonormal."""
    h4 = 1.0 - 2.0 * torch.eye(4, dtype=torch.float64, device=x.device).flip(1)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return (x.view(-1, 256) @ h.t() / 16).view_as(x)


def _mx(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """MX blocks of 32: E4M3 values and their E8M0 exponent bytes."""
    blocks = x.float().view(x.shape[0], -1, 32)
    amax = blocks.abs().amax(-1)
    power = torch.where(amax > 0, torch.ceil(torch.log2(_over(amax, 448))), torch.full_like(amax, -127.0))
    byte = (power + 127).clamp(0, 254)
    q = (blocks / torch.exp2(byte - 127)[..., None]).clamp(-448, 448)
    return q.view(x.shape[0], -1).to(E4M3), byte.to(torch.uint8)


def _blocks(v: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    """v [R, K] times its block scales [R, blocks], float64."""
    return (v.double().view(v.shape[0], scale.shape[1], -1) * scale.double()[..., None]).view(v.shape)


def _unpacked(packed: torch.Tensor) -> torch.Tensor:
    return torch.stack((packed & 15, packed >> 4), -1).view(packed.shape[0], -1).long()


def _e2m1(codes: torch.Tensor) -> torch.Tensor:
    table = torch.tensor([*E2M1, *(-v for v in E2M1)], dtype=torch.float64, device=codes.device)
    return table[codes]


def _int4(v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    groups = v.view(v.shape[0], -1, 64)
    scale = _over(groups.abs().amax(-1), 7).half()
    q = (groups / scale.float()[..., None]).round().clamp(-8, 7)
    return torch.where(scale[..., None] == 0, 0.0, q.double()).view(v.shape), scale


def _weight64(fmt: str, parts: dict) -> torch.Tensor:
    """A stored weight's values, float64 [N, K]."""
    if fmt in ("int8", "fp8"):
        return parts["weight"].double() * parts["scale"].double()[:, None]
    if fmt == "mxfp8":
        return _blocks(parts["weight"].double(), torch.exp2(parts["scale"].double() - 127))
    codes = _unpacked(parts["weight"])
    if fmt == "w4a8":
        level = parts["codebook"][codes].view(codes.shape[0], -1, 16) * parts["group_scale"].float()[..., None]
        return level.round().clamp(-127, 127).double().view(codes.shape) * parts["scale"].double()[:, None]
    if fmt == "svdq_int4":
        return _blocks(codes - 16 * (codes >= 8).long(), parts["scale"])
    return _blocks(_e2m1(codes), parts["scale"].float()) * parts["scale_2"].double()


def _operand64(fmt: str, x: torch.Tensor, parts: dict) -> torch.Tensor:
    """The activation the product sees, float64 [M, K]: x quantized as the format says."""
    if fmt in ("int8", "w4a8"):
        r = _rotated(x.double()).float()
        scale = _over(r.abs().amax(1, keepdim=True), 127).clamp(min=1e-12)
        return (r / scale).round().clamp(-127, 127).double() * scale.double()
    if fmt == "fp8":
        v = x.float()
        scale = _over(v.abs().amax(1, keepdim=True), 448).clamp(min=1e-12)
        return (v / scale).clamp(-448, 448).to(E4M3).double() * scale.double()
    if fmt == "mxfp8":
        q, byte = _mx(x)
        return _blocks(q.double(), torch.exp2(byte.double() - 127))
    if fmt == "nvfp4":
        return x.double()
    smooth = (x.float() * parts["pre_quant_scale"]).bfloat16().float()
    if fmt == "svdq_int4":
        return _blocks(*_int4(smooth))
    g = _over((x.abs().amax(0).float() * parts["pre_quant_scale"]).amax(), 448 * 6)
    groups = smooth.view(x.shape[0], -1, 16)
    scale = (groups.abs().amax(-1) / (6 * g)).clamp(2.0**-9, 448).to(E4M3)
    a = (groups / (scale.float() * g)[..., None]).abs()
    code = torch.zeros_like(a, dtype=torch.long)
    # Ties to the even code.
    for bound, inclusive in ((0.25, False), (0.75, True), (1.25, False), (1.75, True), (2.5, False),
                             (3.5, True), (5.0, False)):  # fmt: skip
        code += (a >= bound) if inclusive else (a > bound)
    code += 8 * (groups < 0)
    return _blocks(_e2m1(code).view(x.shape), scale.float()) * g.double()


def exact(case: dict, seed: int):
    if case["kind"] == "bake":
        return None  # codes and bits, compared as they are
    drawn, fmt = _drawn(case, seed), case["format"]
    outs = []
    for v in drawn.linears:
        x = v.x
        if drawn.tables is not None:
            scale, shift = (t.double() for t in drawn.tables)
            x = x.double()
            centred = x - x.mean(1, keepdim=True)
            x = centred * torch.rsqrt(centred.square().mean(1, keepdim=True) + 1e-6) * (1 + scale) + shift
        y = _operand64(fmt, x, v.parts) @ _weight64(fmt, v.parts).t()
        if case["rank"]:
            low = (v.x.double() @ v.parts["lowrank_down"].to(v.x.dtype).double().t()).bfloat16().double()
            y = y + low @ v.parts["lowrank_up"].double().t()
        outs.append(y if v.bias is None else y + v.bias.double())
    return outs if case["kind"] == "step" else outs[0]
