"""The work a user of this package has it do, as cases that can be timed and compared.

A case is one pass through the public entry points: a forward (inference) or a forward and backward (training step) of
the gated convolution on separate tensors ("operator"), of the Hyena-MR module ("module"), of the convolutional part of
a hyena layer from the dense projection's output on ("mixer"), or of the short-filter operator on time-major operands
("short_hyena").  ``listed()`` holds the named ones, ``draw()`` makes more over the same ranges.

Fields: entry, hl (taps; at most 8 is Hyena-SE, more is Hyena-MR), step (forward+backward), bs, L, g (filter groups),
dg (channels per group), dtype (of the tensors), arith (``cgcg_dtype``: filter and arithmetic), planar (layout of the
projected features: "(p g dg)" instead of "(g dg p)").
"""
import math

import torch

from savanna_amd import two_pass_chunked_gate_conv_gate
from savanna_amd.kernels.cgcg.src.kernel_utils import FwdKernelConfigRefactor
from savanna_amd.kernels.short_hyena import run_short_hyena
from savanna_amd.operators.hyena import CgcgConfig, HyenaMixer, HyenaMROperator, HyenaSEOperator

DEVICE = "cuda:0"
FWD_CFG = FwdKernelConfigRefactor(CHUNK_SIZE=128, BLOCK_D=16, THREADBLOCK_SWIZZLE="row")
BYTES = {"float32": 4, "bfloat16": 2, "float16": 2}


def _case(entry, hl, step, bs, L, g, dg, dtype="bfloat16", arith=None, planar=False, name=None):
    c = {"entry": entry, "hl": hl, "step": step, "bs": bs, "L": L, "g": g, "dg": dg, "dtype": dtype,
         "arith": arith or dtype, "planar": planar}
    return dict({"name": name}, **c) if name else c


def listed():
    return [
        # Hyena-SE forward on a tensor that is hardly more than a launch (the smallest benchmark configuration)
        _case("operator", 7, False, 1, 2048, 16, 16, "float32", name="se_forward_small"),
        # prefill of a short prompt through a Hyena-MR layer of the 7B width: a length no tile divides, no gradients
        _case("mixer", 128, False, 1, 701, 256, 16, name="mr_mixer_prefill_short"),
        # Hyena-MR training step of the operator at the 7B layer shape (the headline benchmark)
        _case("operator", 128, True, 2, 8192, 256, 16, name="mr_step_7b"),
        # the same for one tensor-parallel rank's share of a 40B layer: an eighth of its channels
        _case("operator", 128, True, 1, 8192, 64, 16, name="mr_step_tp_rank"),
        # Hyena-MR module in its default precision (fp32 filter and arithmetic on bf16 activations), ragged batch
        _case("module", 128, True, 3, 5003, 160, 16, arith="float32", name="mr_module_default_precision"),
        # Hyena-MR training step on fp32 tensors (parity runs, small models), filter shorter than a chunk
        _case("operator", 64, True, 2, 4096, 128, 16, "float32", name="mr_step_fp32"),
        # Hyena-MR with groups narrower than a matrix tile: 256 groups on a narrow model
        _case("operator", 128, True, 1, 4096, 256, 8, name="mr_step_narrow_groups"),
        # the short operator on (seqlen, bs, g, dg) operands, the shape its own test uses
        _case("short_hyena", 7, True, 16, 8192, 48, 16, name="short_hyena_step"),
        # convolutional part of a 7B Hyena-MR layer, training step, bf16 arithmetic
        _case("mixer", 128, True, 2, 8192, 256, 16, name="mr_mixer_step_7b"),
        # the same in the default precision
        _case("mixer", 128, True, 2, 8192, 256, 16, arith="float32", name="mr_mixer_step_7b_default_precision"),
        # convolutional part of a 40B Hyena-SE layer, training step
        _case("mixer", 7, True, 1, 32768, 512, 16, name="se_mixer_step_40b"),
        # Hyena-MR forward over a million tokens (long-context prefill)
        _case("operator", 128, False, 1, 1048576, 256, 16, name="mr_forward_1m"),
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case.  Lengths and widths are spread over their logarithm; a training step holds at most 2^27 and a
    forward 2^29 elements per tensor, the narrow groups and long filters of "general" a sixteenth of that."""
    family = rng.choice(["small", "operator_mr", "operator_se", "module", "general", "short_hyena", "mixer_mr",
                         "mixer_mr", "mixer_se", "prefill", "forward_long"])
    dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float32"])
    step = rng.random() < 0.7
    mr = rng.choice([128, 128, 64, rng.randint(9, 128)])
    se = rng.choice([7, 7, 4, rng.randint(2, 8)])
    dg = rng.choice([16, 16, 16, 32])
    cap = 1 << 27 if step else 1 << 29

    def sizes(L_lo, L_hi, d_lo=256, d_hi=8192, bs_hi=8, width=dg, limit=cap):
        g = max(1, _loguniform(rng, d_lo, d_hi) // width)
        bs = _loguniform(rng, 1, bs_hi)
        L = _loguniform(rng, L_lo, L_hi)
        return bs, max(1, min(L, limit // (bs * g * width))), g, width

    arith = rng.choice([dtype, "float32"])
    planar = rng.random() < 0.3
    if family == "small":
        return _case("operator", rng.choice([se, mr]), step, *sizes(64, 2048, 128, 1024, 2), dtype)
    if family == "operator_mr":
        return _case("operator", mr, step, *sizes(512, 65536), dtype)
    if family == "operator_se":
        return _case("operator", se, step, *sizes(512, 65536), dtype)
    if family == "module":
        return _case("module", mr, step, *sizes(512, 65536), dtype, arith)
    if family == "general":
        width, hl = rng.choice([(rng.randint(1, 15), mr), (8, 128), (24, mr), (16, rng.randint(129, 256))])
        return _case("operator", hl, step, *sizes(256, 16384, 128, 4096, 4, width, 1 << 23), dtype)
    if family == "short_hyena":
        return _case("short_hyena", se, step, *sizes(512, 16384, 256, 4096, 16), dtype)
    if family == "mixer_mr":
        return _case("mixer", mr, step, *sizes(512, 65536), dtype, arith, planar)
    if family == "mixer_se":
        return _case("mixer", se, step, *sizes(512, 65536), dtype, arith, planar)
    if family == "prefill":
        return _case("mixer", rng.choice([se, mr]), False, *sizes(16, 2048, 1024, 8192, 2), dtype, arith, planar)
    return _case("operator", rng.choice([se, mr]), False, *sizes(65536, 524288, 1024, 4096, 1), rng.choice(["bfloat16", "float16"]))


def _normal(shape, dtype, gen):
    """N(0, 1) values, drawn in the type itself (a large 16-bit tensor needs no fp32 copy)."""
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=gen)


def _filter(c, gen):
    """(g, 1, hl) fp32: N(0, 1/hl), with an exponential decay of log-uniform rate for Hyena-MR."""
    g, hl = c["g"], c["hl"]
    h = torch.randn(g, hl, generator=gen, device=DEVICE) / math.sqrt(hl)
    if hl > 8:
        lo, hi = math.log(1e-3), math.log(1e-1)
        rate = torch.exp(lo + (hi - lo) * torch.rand(g, 1, generator=gen, device=DEVICE))
        h = h * torch.exp(-rate * torch.arange(hl, device=DEVICE))
    return h.unsqueeze(1)


def _module(c, gen):
    """The operator module with the weights a trained layer would have (no tiny initialisation)."""
    cfg = CgcgConfig(cgcg_dtype=c["arith"])
    hidden = c["g"] * c["dg"]
    if c["hl"] > 8:
        op = HyenaMROperator(hidden, c["g"], c["hl"], cfg, small_init=False, device=DEVICE)
        with torch.no_grad():
            op.filter.h.copy_(torch.randn(op.filter.h.shape, generator=gen, device=DEVICE) / math.sqrt(c["hl"]))
    else:
        op = HyenaSEOperator(hidden, c["g"], c["hl"], cfg, device=DEVICE)
        with torch.no_grad():
            op.short_conv_weight.copy_(_filter(c, gen))
    return op


def prepare(c, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = getattr(torch, c["dtype"])
    bs, L, g, dg, step = c["bs"], c["L"], c["g"], c["dg"], c["step"]
    s = {"case": c, "params": []}
    if c["entry"] == "mixer":
        mixer = HyenaMixer(_module(c, gen), 3, dtype=dtype, device=DEVICE, interleave_projections=not c["planar"])
        w = mixer.hyena_proj_conv.short_conv_weight
        with torch.no_grad():
            w.copy_((2 * torch.rand(w.shape, generator=gen, device=DEVICE) - 1) / math.sqrt(3))
        s["fn"], s["inputs"] = mixer, [_normal((bs, L, 3 * g * dg), dtype, gen)]
        s["params"] = list(mixer.parameters())
    elif c["entry"] == "module":
        s["fn"] = _module(c, gen)
        s["inputs"] = [_normal((bs, L, g, dg), dtype, gen) for _ in range(3)]
        s["params"] = list(s["fn"].parameters())
    elif c["entry"] == "short_hyena":
        s["inputs"] = [_normal((L, bs, g, dg), dtype, gen) for _ in range(3)] + [_filter(c, gen).to(dtype)]
    else:
        s["inputs"] = [_normal((bs, L, g, dg), dtype, gen) for _ in range(3)] + [_filter(c, gen).to(dtype)]
    if step:
        for t in s["inputs"]:
            t.requires_grad_(True)
        s["dy"] = _normal((bs, L, g * dg), dtype, gen)
    return s


def _forward(s):
    """(bs, L, g * dg), the layout in which the output projection reads it."""
    c, inputs = s["case"], s["inputs"]
    bs, L, g, dg = c["bs"], c["L"], c["g"], c["dg"]
    if c["entry"] in ("mixer", "module"):
        return s["fn"](*inputs)
    if c["entry"] == "short_hyena":
        q, k, v, w = inputs
        return run_short_hyena(q, k, v, w, autotune=True).permute(0, 2, 1, 3).reshape(bs, L, g * dg)
    x, B, C, h = inputs
    y = two_pass_chunked_gate_conv_gate(x, B, C, h, bs, L, g, dg, fwd_kernel_cfg=FWD_CFG)
    return y.reshape(bs, L, g * dg)


def run(s):
    if not s["case"]["step"]:
        with torch.no_grad():
            return _forward(s)
    y = _forward(s)
    return [y.detach(), *torch.autograd.grad(y, s["inputs"] + s["params"], s["dy"])]


def work(c):
    """Bytes: forward reads three tensors and writes one, backward reads those and dy and writes three gradients;
    filters and their gradients once.  Flops: two per tap and sample, for the forward, the input gradient and the
    filter gradient; the featurizer of a mixer is three taps on each of the three operands."""
    n, step = c["bs"] * c["L"] * c["g"] * c["dg"], c["step"]
    filt = c["g"] * c["hl"] * BYTES[c["arith"]]
    taps = c["hl"]
    if c["entry"] == "mixer":
        filt += 3 * c["g"] * c["dg"] * 3 * BYTES[c["dtype"]]
        taps += 9
    return {"bytes": (11 if step else 4) * n * BYTES[c["dtype"]] + (3 if step else 1) * filt,
            "flops": (3 if step else 1) * 2 * n * taps}


def tolerance(c):
    """Relative error in the 2-norm, three to five times what the package shows against fp64 on the same inputs: fp32
    4.5e-7 over 1400 rows, growing with the rows that a filter gradient sums; 16-bit arithmetic, which rounds gated
    products and a mixer's features to the type, 2.3e-3 to 4.1e-3 in bf16 and 2.9e-4 to 5.0e-4 in f16; fp32 arithmetic on
    16-bit operands, whose results are rounded once, 2.1e-4 and 3.4e-5 against the rounded exact ones."""
    if c["dtype"] == "float32":
        return {"rel": 1e-5}
    once = c["arith"] == "float32" and c["entry"] != "mixer"
    return {"rel": {"bfloat16": (1e-2, 1e-3), "float16": (2e-3, 1.5e-4)}[c["dtype"]][once]}
