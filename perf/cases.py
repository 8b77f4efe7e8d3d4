"""What a user of this package has it do, as cases that can be timed.

Each case is a plain dict; its "op" names the public entry point:

  linear      an ``RNSLinear`` forward (activation quantization, product,
              dequantization) on a layer whose weight is prepared
  product     ``HipRNSBackend.matmul_prepared_fused``: integer activations
              against a prepared weight, exact int64 out
  adaptive    ``matmul_prepared_adaptive_fused``: the same with the channel
              prefix chosen from the activations
  requests    ``matmul_prepared_fused_requests``: continuous batching, a few
              requests of a few rows each in one merged call
  unprepared  ``matmul_wide``: both operands plain integers, encoded in the
              call (what a program does with a matrix it multiplies once)

Sizes: 768 x 2304 is the fused query/key/value projection of OPT-125m and
768 x 768 its output projection, 4096 x 12288 the fused projection of
OPT-6.7B; 4096 tokens are a batch of 8 sequences of 512.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "rns-llm_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from rns_llm_amd import HipRNSBackend, RNSLinear, choose_moduli_for_dot  # noqa: E402

DEVICE = "cuda"
FLOATS = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
# the work of the largest listed case (channels x M x K x N)
LARGEST = 4 * 2048 * 4096 * 12288


def listed() -> list[dict]:
    return [
        # one new token through a fused projection layer: launches and host time
        dict(name="linear 1 token", op="linear", m=1, k=768, n=2304, bits=8, dtype="float16", bias=True, packed=False),
        # a prefill batch, 8 sequences of 512 tokens, through the same layer
        dict(name="linear 4096 tokens", op="linear", m=4096, k=768, n=2304, bits=8, dtype="float16", bias=True,
             packed=False),
        # a 12-bit layer of odd sizes: K no multiple of the 64-byte step, N odd, a short prompt
        dict(name="linear 12-bit ragged", op="linear", m=77, k=1000, n=1531, bits=12, dtype="bfloat16", bias=True,
             packed=False),
        # decode with four requests of one row each merged into one call
        dict(name="requests 4 x 1", op="requests", m=4, each=1, k=768, n=768, bits=8),
        # the package's headline call: 256 tokens, int8, exact int64 out
        dict(name="int8 256 tokens", op="product", m=256, k=768, n=2304, bits=8, packed=False),
        # decode of one token against a large projection: streaming the weight
        dict(name="int8 wide 1 token", op="product", m=1, k=4096, n=12288, bits=8, packed=False),
        # prefill against a large projection: the largest product
        dict(name="int8 wide 2048 tokens", op="product", m=2048, k=4096, n=12288, bits=8, packed=False),
        # the same with a shorter channel prefix, which activations with a few
        # large features (as transformers have) allow
        dict(name="adaptive wide 512 tokens", op="adaptive", m=512, k=4096, n=12288, bits=8, outliers=True),
        # 16-bit weights and activations as six residue planes, prefill
        dict(name="int16 wide 512 tokens", op="product", m=512, k=4096, n=12288, bits=16, packed=False),
        # 16-bit weights kept in two bytes per value: a small decode batch
        dict(name="packed wide 4 tokens", op="product", m=4, k=4096, n=12288, bits=16, packed=True),
        # ... and prefill
        dict(name="packed wide 512 tokens", op="product", m=512, k=4096, n=12288, bits=16, packed=True),
        # two int8 matrices multiplied once: encode, repack, product, decode
        dict(name="unprepared 256 x 2048", op="unprepared", m=256, k=2048, n=2048, bits=8),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng: random.Random, lo: int, hi: int) -> int:
    """A layer width: two in three times a multiple of 64, as model widths
    are, otherwise any number."""
    v = _log(rng, lo, hi)
    return max(lo, v // 64 * 64) if rng.random() < 0.67 else v


def draw(rng: random.Random) -> dict:
    op = rng.choice(["linear", "linear", "linear", "product", "product", "product", "product", "adaptive", "requests",
                     "unprepared"])
    k, n = _size(rng, 512, 4096), _size(rng, 512, 12288)
    if op == "requests":
        each, count = rng.randint(1, 8), rng.randint(2, 8)
        return dict(op=op, m=each * count, each=each, k=k, n=n, bits=8)
    bits = 8 if op in ("adaptive", "unprepared") else rng.choice([8, 8, 8, 12, 16, 16])
    packed = bits > 8 and rng.random() < 0.6
    most = LARGEST // (len(_moduli(k, bits)) * k * n)
    if op == "unprepared":
        n = min(n, 4096)
    m = min(_log(rng, 1, 4096), max(1, most))
    if op == "linear":
        return dict(op=op, m=m, k=k, n=n, bits=bits, dtype=rng.choice(["float16", "bfloat16", "float32"]),
                    bias=rng.random() < 0.7, packed=packed)
    if op == "adaptive":
        return dict(op=op, m=m, k=k, n=n, bits=bits, outliers=rng.random() < 0.5)
    if op == "unprepared":
        return dict(op=op, m=m, k=k, n=n, bits=bits)
    return dict(op=op, m=m, k=k, n=n, bits=bits, packed=packed)


def _moduli(k: int, bits: int) -> tuple[int, ...]:
    most = 2 ** (bits - 1) - 1
    return choose_moduli_for_dot(k, most, most, strategy="dense_coprime")


def _quantize(values: torch.Tensor, bits: int) -> torch.Tensor:
    """Symmetric quantization of each row."""
    most = 2 ** (bits - 1) - 1
    scale = values.abs().amax(dim=1, keepdim=True) / most
    return torch.clamp(torch.round(values / scale), -most, most).to(torch.int8 if bits == 8 else torch.int16)


def _inputs(case: dict, seed: int):
    """Activations [M, K] as a layer norm leaves them (unit variance) and the
    weight [N, K] as a projection has it, in float32, from the seed alone."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    x = torch.randn((case["m"], case["k"]), generator=gen, device=DEVICE)
    if case.get("outliers"):
        # 16 features some 24 times the others', the same in every token
        x[:, torch.randperm(case["k"], generator=gen, device=DEVICE)[:16]] *= 24.0
    w = torch.randn((case["n"], case["k"]), generator=gen, device=DEVICE) * 0.02
    return x, w, gen


def prepare(case: dict, seed: int) -> dict:
    backend = HipRNSBackend()
    x, w, gen = _inputs(case, seed)
    m, k, n, bits = case["m"], case["k"], case["n"], case["bits"]
    state = {"op": case["op"], "backend": backend}
    if case["op"] == "linear":
        dtype = FLOATS[case["dtype"]]
        with torch.device(DEVICE):
            layer = RNSLinear(k, n, bias=case["bias"], backend=backend, mode="rns", quant_bits=bits,
                              packed_weights=case["packed"]).to(dtype=dtype).eval()
        with torch.no_grad():
            layer.weight.copy_(w)
            if case["bias"]:
                layer.bias.copy_(torch.randn((n,), generator=gen, device=DEVICE) * 0.1)
        layer.prepare_weight()
        state.update(layer=layer, x=x.to(dtype))
        return state
    moduli = _moduli(k, bits)
    a, w = _quantize(x, bits), _quantize(w, bits)
    if case["op"] == "unprepared":
        state.update(a=a, b=w.t().contiguous(), moduli=moduli)
        return state
    if case["op"] == "requests":
        rows = [case["each"]] * (m // case["each"])
        state.update(requests=[r.contiguous() for r in a.split(case["each"])],
                     weight=backend.prepare_weight_nk(w, moduli),
                     workspace=backend.create_request_batch_workspace(
                         device=a.device, dtype=a.dtype, rows_per_request=rows, k=k, channels=len(moduli), n=n))
        return state
    workspace = backend.create_workspace(device=a.device, channels=len(moduli), m=m, n=n, k=k)
    if case["op"] == "adaptive":
        state.update(weight=backend.prepare_weight_adaptive_nk(w, moduli, min_channels=min(3, len(moduli))), a=a,
                     workspaces={len(moduli): workspace})
    else:
        prepare_nk = backend.prepare_weight_packed_nk if case["packed"] else backend.prepare_weight_nk
        state.update(weight=prepare_nk(w, moduli), a=a, workspace=workspace)
    return state


def run(state: dict):
    op = state["op"]
    if op == "linear":
        with torch.no_grad():
            return state["layer"](state["x"])
    backend = state["backend"]
    if op == "product":
        return backend.matmul_prepared_fused(state["a"], state["weight"], workspace=state["workspace"])
    if op == "adaptive":
        out, meta = backend.matmul_prepared_adaptive_fused(
            state["a"], state["weight"], workspace_by_channels=state["workspaces"], return_metadata=True)
        return out, meta.device_tensor
    if op == "requests":
        return backend.matmul_prepared_fused_requests(state["requests"], state["weight"], workspace=state["workspace"])
    return backend.matmul_wide(state["a"], state["b"], state["moduli"])


def work(case: dict) -> dict:
    m, k, n, bits = case["m"], case["k"], case["n"], case["bits"]
    channels = len(_moduli(k, bits))
    if case.get("outliers"):
        channels = min(channels, 3)  # the prefix such activations need
    value = 1 if bits == 8 else 2
    if case["op"] == "linear":
        a = out = FLOATS[case["dtype"]].itemsize
    else:
        a, out = value, 8
    # a prepared weight is one byte per residue channel, a packed one two
    # bytes per value, an unprepared one the plain integers
    packed = case.get("packed", False)
    weight = value if case["op"] == "unprepared" else 2 if packed else channels
    # a product per residue channel; of packed 16-bit weights no more than a
    # product per pair of their bytes and the activations'
    products = min(channels, 2 * value) if packed else channels
    return {"bytes": a * m * k + weight * k * n + out * m * n, "flops": 2 * products * m * k * n}


def tolerance(case: dict):
    """Integer outputs are exact.  A layer's differ from the 64-bit result by
    the rounding to their type (rel 3.4e-4 seen in float16, 1.7e-3 in
    bfloat16) or, in float32 (2.2e-6), by the float32 scales and by the few
    activations that lie within float32 rounding of the middle between two
    quantized values and may go either way; stated is about four times what
    was seen, more in float32 for those ties at 8 bits."""
    if case["op"] != "linear":
        return "exact"
    return {"rel": {"float16": 1.3e-3, "bfloat16": 7e-3, "float32": 2e-5}[case["dtype"]]}


def exact(case: dict, seed: int):
    x, w, gen = _inputs(case, seed)
    bits = case["bits"]
    most = 2 ** (bits - 1) - 1
    if case["op"] == "linear":
        dtype = FLOATS[case["dtype"]]
        bias = torch.randn((case["n"],), generator=gen, device=DEVICE) * 0.1
        x, w = x.to(dtype).double(), w.to(dtype).double()
        s_x = x.abs().amax() / most
        s_w = w.abs().amax(dim=1, keepdim=True) / most
        q_x, q_w = torch.round(x / s_x).clamp(-most, most), torch.round(w / s_w).clamp(-most, most)
        y = (q_x @ q_w.t()) * s_x * s_w.t()
        return y + bias.to(dtype).double() if case["bias"] else y
    # every partial sum is an integer below 2^53: float64 products are exact
    y = (_quantize(x, bits).double() @ _quantize(w, bits).double().t()).to(torch.int64)
    if case["op"] == "requests":
        return tuple(y.split(case["each"]))
    return (y, None) if case["op"] == "adaptive" else y
