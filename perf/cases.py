"""The work a user of this framework has it do, as cases that can be timed.

Four kinds of call, each through the package binding (`l2c`) and the C ABI
below it, over the sizes that the harness, the applications and the tests use
(batch 1 to 1024, rows of 288 to 16384 values, 288 to 11008 matrix rows):

  iteration  one llama2c iteration in fp32: rmsnorm and softmax of every
             vector and the W.x product, as three launches with the
             matrix-vector product ("separate"), as the one fused launch
             ("fused"), or with the batched contraction ("batched")
  product    the quantized-weight contraction of bf16 activations: "mxfp4" and
             "fp8" on the exact path, "mxfp4s" and "fp8s" with the activations
             quantized to MXFP8 on the way
  step       one step of the greedy decoder over `batch` sequences, with the
             classifier in "fp32", "bf16", "mxfp6" or "nvfp4": rmsnorm of each
             sequence's embedding row, the conversion of the result, the
             logits, softmax and argmax
  quantize   a weight matrix into one of the formats, when a model is loaded

`size` is the contraction's length and `rows` the matrix's rows (a step's
width and vocabulary).
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cuda-elastic_amd"))
import l2c  # noqa: E402

EPS = l2c.RMS_EPSILON
LARGEST = 1024 * 16384 * 8192  # batch x size x rows of the largest listed case


def _case(kind, form, batch, size, rows, name=None):
    c = {"kind": kind, "form": form, "batch": batch, "size": size, "rows": rows}
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smoke iteration of the tests and the bench: nothing but launches.
        _case("iteration", "separate", 1, 288, 288, "iteration_1x288x288"),
        # The launch-bound small batch of the bench, with every vector multiplied.
        _case("iteration", "batched", 8, 768, 2048, "batched_8x768x2048"),
        # One decoded token of a 4096-wide layer: a 172 MiB matrix streamed once.
        _case("iteration", "fused", 1, 4096, 11008, "fused_1x4096x11008"),
        # A ragged batch whose rows are no multiple of four values.
        _case("iteration", "batched", 130, 5003, 1501, "batched_130x5003x1501"),
        # The headline: the largest profiled shape.
        _case("iteration", "batched", 1024, 16384, 8192, "batched_1024x16384x8192"),
        # Decode of sixteen sequences with 4-bit weights.
        _case("product", "mxfp4", 16, 4096, 11008, "mxfp4_16x4096x11008"),
        # A prefill chunk, or a full decode batch, with 8-bit weights.
        _case("product", "fp8", 256, 4096, 11008, "fp8_256x4096x11008"),
        # The benchmark's quantized shape on the block-scaled matrix cores.
        _case("product", "mxfp4s", 1024, 16384, 8192, "mxfp4s_1024x16384x8192"),
        # The decoder application at its own precision, a middling batch.
        _case("step", "fp32", 64, 2048, 8192, "step_fp32_64x2048x8192"),
        # A ragged decode batch with the bf16 classifier.
        _case("step", "bf16", 40, 4096, 8004, "step_bf16_40x4096x8004"),
        # The low-precision classifier experiment's large preset.
        _case("step", "nvfp4", 1024, 16384, 8192, "step_nvfp4_1024x16384x8192"),
        # Weights of one layer quantized at load.
        _case("quantize", "mxfp4", 1, 4096, 11008, "quantize_mxfp4_11008x4096"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("iteration",) * 3 + ("product",) * 3 + ("step",) * 3 + ("quantize",))
    batch, size, rows = _log_int(rng, 1, 1024), _log_int(rng, 288, 16384), _log_int(rng, 288, 11008)
    # Four sizes in ten are a model's (multiples of 256), the rest whatever the format takes.
    granule = 256 if rng.random() < 0.4 else 1
    if kind == "iteration":
        form = rng.choice(("separate", "fused", "batched", "batched"))
    elif kind == "product":
        form = rng.choice(("mxfp4", "fp8", "mxfp4s", "fp8s"))
        granule = max(granule, 128 if form.endswith("s") else 32)
    elif kind == "step":
        form = rng.choice(("fp32", "bf16", "mxfp6", "nvfp4"))
        granule = max(granule, {"fp32": 1, "bf16": 32, "mxfp6": 128, "nvfp4": 32}[form])
    else:
        form = rng.choice(("mxfp4", "fp8", "mxfp6", "nvfp4"))
        granule = max(granule, {"mxfp4": 32, "fp8": 1, "mxfp6": 128, "nvfp4": 16}[form])
        batch = 1
    size = max(granule, round(size / granule) * granule)
    if granule == 256:
        rows = max(256, round(rows / 256) * 256)
    while batch * size * rows > LARGEST:
        batch = batch // 2
    return _case(kind, form, max(1, batch), size, rows)


# ---------------------------------------------------------------------------
# Inputs: the bench's distributions, from the seed alone.

def _inputs(case, seed):
    """The fp32 tensors of a case."""
    batch, size, rows = case["batch"], case["size"], case["rows"]
    gen = torch.Generator("cuda").manual_seed(seed)

    def uniform(*shape, low=-1.0, high=1.0):
        return torch.empty(*shape, device="cuda").uniform_(low, high, generator=gen)

    def normal(*shape):
        return torch.empty(*shape, device="cuda").normal_(generator=gen)

    if case["kind"] == "iteration":
        return {"x": uniform(batch, size), "logits": uniform(batch, size), "weight": uniform(size, low=0.5, high=1.5),
                "W": uniform(rows, size).div_(math.sqrt(size))}
    if case["kind"] == "step":
        return {"tokens": torch.randint(rows, (batch,), generator=gen, device="cuda", dtype=torch.int32),
                "embedding": normal(rows, size), "weight": uniform(size, low=0.5, high=1.5),
                "W": normal(rows, size).div_(math.sqrt(size))}
    d = {"W": normal(rows, size).div_(math.sqrt(size))}
    if case["kind"] == "product":
        d["x"] = uniform(batch, size)
    return d


def _u8(n):
    return torch.empty(n, dtype=torch.uint8, device="cuda")


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _bf16(n):
    return torch.empty(n, dtype=torch.int16, device="cuda")


def _quantized(form, rows, size):
    """Buffers of one quantized [rows][size] operand."""
    if form.startswith("mxfp4"):
        return {"codes": _u8(rows * size // 2), "scales": _u8(rows * size // 32)}
    if form.startswith("fp8"):
        return {"codes": _u8(rows * size), "scales": _f32(rows)}
    if form == "mxfp6":
        codes, scales = l2c.mxfp6_bytes(rows, size)
        return {"codes": _u8(codes), "scales": _u8(scales)}
    if form == "nvfp4":
        return {"codes": _u8(rows * size // 2), "scales": _u8(rows * size // 16), "tensor_scales": _f32(2)}
    return {}


def _quantize(form, q, W, rows, size, partials=None, expanded=None):
    if form.startswith("mxfp4"):
        l2c.quantize_mxfp4(q["codes"], q["scales"], W, rows, size)
    elif form.startswith("fp8"):
        l2c.quantize_fp8(q["codes"], q["scales"], W, rows, size)
    elif form == "mxfp6":
        l2c.quantize_mxfp6(q["codes"], q["scales"], W, rows, size)
    else:
        l2c.nvfp4_tensor_scales(q["tensor_scales"], W, rows * size, partials)
        l2c.quantize_nvfp4(q["codes"], q["scales"], W, q["tensor_scales"], rows, size, expanded=expanded)


def prepare(case, seed):
    kind, form, batch, size, rows = (case[k] for k in ("kind", "form", "batch", "size", "rows"))
    s = dict(case, **_inputs(case, seed))
    if kind == "iteration":
        s.update(normalized=_f32(batch, size), softmax=_f32(batch, size),
                 product=_f32(batch, rows) if form == "batched" else _f32(rows))
        return s
    if kind == "quantize":
        s["q"] = _quantized(form, rows, size)
        s["partials"] = _f32(l2c.NVFP4_PARTIALS)
        return s
    s["q"] = q = _quantized(form, rows, size)
    if kind == "product":
        _quantize(form, q, s.pop("W"), rows, size)
        x = s.pop("x")
        s["xbf16"] = _bf16(batch * size)
        l2c.to_bf16(s["xbf16"], x, batch * size)
        if form.endswith("s"):
            s["workspace"] = _u8(l2c.mxfp8_workspace_bytes(batch, size))
        s["out"] = _f32(batch, rows)
        return s
    s.update(normalized=_f32(batch, size), out=_f32(batch, rows), probabilities=_f32(batch, rows),
             next=torch.empty(batch, dtype=torch.int32, device="cuda"),
             generated=torch.empty(batch, dtype=torch.int32, device="cuda"))
    if form == "bf16":
        s.update(wbf16=_bf16(rows * size), xbf16=_bf16(batch * size))
        l2c.to_bf16(s["wbf16"], s.pop("W"), rows * size)
    elif form == "mxfp6":
        s["xq"] = _quantized(form, batch, size)
        _quantize(form, q, s.pop("W"), rows, size)
    elif form == "nvfp4":
        s.update(wbf16=_bf16(rows * size), xbf16=_bf16(batch * size), xq=_quantized(form, batch, size),
                 partials=_f32(l2c.NVFP4_PARTIALS), alpha=_f32(1))
        _quantize(form, q, s.pop("W"), rows, size, s["partials"], s["wbf16"])
    return s


# ---------------------------------------------------------------------------
# One pass.

def _run_iteration(s):
    form, batch, size, rows = s["form"], s["batch"], s["size"], s["rows"]
    if form == "fused":
        l2c.fused(s["normalized"], s["x"], s["weight"], s["softmax"], s["logits"], s["product"], s["W"], size, batch,
                  batch, rows)
    else:
        l2c.rmsnorm(s["normalized"], s["x"], s["weight"], size, batch)
        l2c.softmax(s["softmax"], s["logits"], size, batch)
        if form == "batched":
            l2c.matmul(s["product"], s["x"], s["W"], batch, size, rows)
        else:
            l2c.matvec(s["product"], s["x"], s["W"], size, rows)
    return {"normalized": s["normalized"], "softmax": s["softmax"], "product": s["product"]}


def _run_product(s):
    q, form = s["q"], s["form"]
    fmt = l2c.Q_MXFP4 if form.startswith("mxfp4") else l2c.Q_FP8
    if form.endswith("s"):
        l2c.matmul_qs(s["out"], s["xbf16"], q["codes"], q["scales"], fmt, s["batch"], s["size"], s["rows"],
                      s["workspace"])
    else:
        l2c.matmul_q(s["out"], s["xbf16"], q["codes"], q["scales"], fmt, s["batch"], s["size"], s["rows"])
    return s["out"]


def _run_step(s):
    form, batch, size, rows = s["form"], s["batch"], s["size"], s["rows"]
    l2c.decoder_rmsnorm(s["normalized"], s["tokens"], s["embedding"], s["weight"], size, rows, batch)
    if form == "fp32":
        l2c.matmul(s["out"], s["normalized"], s["W"], batch, size, rows)
    elif form == "bf16":
        l2c.to_bf16_x4(s["xbf16"], s["normalized"], batch * size)
        l2c.matmul_bf16(s["out"], s["xbf16"], s["wbf16"], batch, size, rows)
    elif form == "mxfp6":
        q, xq = s["q"], s["xq"]
        l2c.quantize_mxfp6(xq["codes"], xq["scales"], s["normalized"], batch, size)
        l2c.matmul_mxfp6(s["out"], xq["codes"], xq["scales"], q["codes"], q["scales"], batch, size, rows)
    else:
        q, xq = s["q"], s["xq"]
        l2c.nvfp4_tensor_scales(xq["tensor_scales"], s["normalized"], batch * size, s["partials"], alpha=s["alpha"],
                                other_decode=q["tensor_scales"][1:])
        l2c.quantize_nvfp4(xq["codes"], xq["scales"], s["normalized"], xq["tensor_scales"], batch, size,
                           expanded=s["xbf16"])
        l2c.matmul_bf16(s["out"], s["xbf16"], s["wbf16"], batch, size, rows, alpha=s["alpha"])
    # The next tokens go to a buffer of their own, so a state can be run again.
    l2c.decoder_softmax_argmax(s["probabilities"], s["out"], s["next"], s["generated"], rows, batch, 1, 0)
    return {"logits": s["out"], "probabilities": s["probabilities"], "next": s["next"], "generated": s["generated"]}


def _run_quantize(s):
    _quantize(s["form"], s["q"], s["W"], s["rows"], s["size"], s["partials"])
    return s["q"]


def run(state):
    return {"iteration": _run_iteration, "product": _run_product, "step": _run_step,
            "quantize": _run_quantize}[state["kind"]](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without.

WEIGHT_BYTES = {"fp32": 4, "bf16": 2, "mxfp4": 0.5 + 1 / 32, "fp8": 1, "mxfp6": 0.75 + 1 / 32, "nvfp4": 0.5 + 1 / 16}


def work(case):
    kind, form, batch, size, rows = (case[k] for k in ("kind", "form", "batch", "size", "rows"))
    vectors = batch * size
    if kind == "quantize":
        return {"bytes": rows * size * (4 + WEIGHT_BYTES[form]), "flops": rows * size}
    if kind == "iteration":
        products = batch if form == "batched" else 1
        # x and the logits in, both results out; the weight; W in, the product out.
        return {"bytes": 4 * (4 * vectors + size + rows * size + products * rows),
                "flops": 2 * products * size * rows + 8 * vectors}
    if kind == "product":
        return {"bytes": 2 * vectors + rows * size * WEIGHT_BYTES[form.rstrip("s")] + 4 * batch * rows,
                "flops": 2 * vectors * rows}
    # A step: the sequences' embedding rows, the weight, W; logits and probabilities out.
    return {"bytes": 4 * vectors + 4 * size + rows * size * WEIGHT_BYTES[form] + 8 * batch * rows,
            "flops": 2 * vectors * rows + 8 * vectors + 4 * batch * rows}


def tolerance(case):
    # Codes and scales are whole numbers (and fp32 row and tensor scales that
    # are single divisions).
    if case["kind"] == "quantize":
        return "exact"
    # A step's rmsnorm summed in another order moves some of its fp32 results by
    # one place, and now and then a code on the other side of a rounding
    # boundary: measured against 64 bits 3e-4 to 5e-4 for the 4- and 6-bit
    # codes, 1e-5 for bf16.
    if case["kind"] == "step" and case["form"] in ("mxfp6", "nvfp4"):
        return {"rel": 2e-3, "differ": 0.01}
    if case["kind"] == "step" and case["form"] == "bf16":
        return {"rel": 1e-4, "differ": 0.01}
    # fp32 sums of exact products: 1e-7 to 2.5e-6 against 64 bits. Tokens are
    # whole values that only a tie within the rounding could move.
    return {"rel": 1e-5, "max": 2e-4, "differ": 0.01}


# ---------------------------------------------------------------------------
# The same in 64 bits.

def _pow2(e):
    """2^e in fp64 from the exponent field (library powers may round)."""
    return (e.long() + 1023).bitwise_left_shift(52).view(torch.float64)


def _minifloat(v, mantissa, lowest, top):
    """v (fp64) to the nearest value of a small float format, ties to even,
    saturating: `mantissa` bits, smallest exponent `lowest`, largest value `top`."""
    a = v.abs()
    exponent = torch.frexp(a)[1].sub(1).clamp_(min=lowest).sub_(mantissa)
    q = (a * _pow2(-exponent)).round_().mul_(_pow2(exponent)).clamp_(max=top)
    return torch.copysign(q, v)


def _e2m1(v):
    return _minifloat(v, 1, 0, 6.0)


def _e3m2(v):
    return _minifloat(v, 2, -2, 28.0)


def _e4m3(v):
    return _minifloat(v, 3, -6, 448.0)


def _block_scaled(x, encode, shift, carry):
    """x (fp32) in blocks of 32 with a shared power of two: the exponent of the
    block's maximum less `shift`, plus one where `carry` says so of its significand in [1, 2)."""
    blocks = x.double().reshape(-1, 32)
    significand, exponent = torch.frexp(blocks.abs().amax(1, keepdim=True))
    e = (exponent - 1 - shift + carry(significand * 2).int()).clamp_(-127, 127)
    return (encode(blocks * _pow2(-e)) * _pow2(e)).reshape(x.shape)


def _mxfp4(x):
    return _block_scaled(x, _e2m1, 3, lambda m: m >= 1.5)


def _mxfp6(x):
    return _block_scaled(x, _e3m2, 4, lambda m: m > 2)


def _mxfp8(x):
    return _block_scaled(x, _e4m3, 8, lambda m: m > 1.75)


def _fp8(x):
    amax = x.abs().amax(1, keepdim=True)
    scale = amax / torch.full_like(amax, 448.0)  # by a tensor: torch multiplies by a number's reciprocal
    return _e4m3((x / scale).double()) * scale.double()


def _nvfp4(x):
    """The values without the tensor scale, and the tensor's decode scale (fp32)."""
    top = x.abs().max()
    s = torch.full_like(top, 2688.0) / top
    blocks = x.reshape(-1, 16)
    amax = blocks.abs().amax(1, keepdim=True)
    f = _e4m3((amax / torch.full_like(amax, 6.0) * s).double()).float()
    codes = _e2m1(torch.where(f > 0, (blocks * s) / f, torch.zeros_like(blocks)).double())
    return (codes * f.double()).reshape(x.shape), torch.ones_like(s) / s


def _rmsnorm64(x, weight):
    x = x.double()
    return x / (x.square().mean(1, keepdim=True) + EPS).sqrt() * weight.double()


def _exact_quantize(case, d):
    """Only fp32 scales are computed numbers; codes and block scales are whole."""
    W = d["W"].double()
    if case["form"] == "fp8":
        return {"codes": None, "scales": W.abs().amax(1) / 448.0}
    if case["form"] == "nvfp4":
        s = 2688.0 / W.abs().max()
        return {"codes": None, "scales": None, "tensor_scales": torch.stack((s, 1.0 / s))}
    return None


def exact(case, seed):
    d = _inputs(case, seed)
    kind, form = case["kind"], case["form"]
    if kind == "quantize":
        return _exact_quantize(case, d)
    if kind == "iteration":
        x = d["x"].double()
        product = x @ d["W"].double().T if form == "batched" else d["W"].double() @ x[0]
        return {"normalized": _rmsnorm64(d["x"], d["weight"]), "softmax": d["logits"].double().softmax(1),
                "product": product}
    if kind == "product":
        W = _mxfp4(d.pop("W")) if form.startswith("mxfp4") else _fp8(d.pop("W"))
        x = d["x"].bfloat16().float()
        return (_mxfp8(x) if form.endswith("s") else x.double()) @ W.T
    normalized = _rmsnorm64(d["embedding"][d["tokens"].long()], d["weight"])
    if form == "fp32":
        logits = normalized @ d["W"].double().T
    elif form == "bf16":
        logits = normalized.float().bfloat16().double() @ d["W"].bfloat16().double().T
    elif form == "mxfp6":
        logits = _mxfp6(normalized.float()) @ _mxfp6(d["W"]).T
    else:
        (xv, xd), (wv, wd) = _nvfp4(normalized.float()), _nvfp4(d["W"])
        logits = (xv @ wv.T) * (xd * wd).double()
    return {"logits": logits, "probabilities": logits.softmax(1), "next": None, "generated": None}
