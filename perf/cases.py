"""Timed cases: what a user of this package has the GPU do, through its public modules.

Four kinds of call, the four levels at which the denoiser is used:

  block      ``SwinLayer.forward``: one Swin layer dropped into somebody else's model, the residual stream in and out
  denoiser   ``LocalAERIS.forward``: one function evaluation of the diffusion sampler, input channels to output channels
  sample     ``TrigFlowSampler.sample``, called eagerly: one draw from the diffusion model, 2 n - 1 denoiser calls
  forecast   ``_Rollout.run`` of ``TrigFlowSampler.begin_rollout``: autoregressive forecast steps replayed as HIP graphs

A case is a dict of plain values; every kind takes the same geometry keys.  ``preset`` "spec" is the classic Swin block
(LayerNorm, relative-position bias, shift mask, GELU MLP, biases), "ref" the reference's own (RMSNorm, six-way modulation
ahead of the norm, SwiGLU, no biases).  Weights are random with unit gain (matrices of standard deviation fan_in^-1/2, so
every branch adds a term as large as the stream, as in a trained model), inputs are standard normal fields, as
per-channel standardised atmospheric fields are.
"""
from __future__ import annotations

import importlib
import math

import torch

amd = importlib.import_module("aeris-gb_amd")

DEVICE = "cuda"
MAX_DRAW_FLOPS = 3.0e14  # a drawn case: at most about a fifth of the full denoiser step


def _case(kind, name, H, W, ws_y, ws_x, dim, heads, head_dim, mlp, preset, **kw):
    c = {"name": name, "kind": kind, "H": H, "W": W, "ws_y": ws_y, "ws_x": ws_x, "dim": dim, "heads": heads,
         "head_dim": head_dim, "mlp": mlp, "preset": preset, "batch": 1, "mod_ways": 3 if preset == "ref" else 2,
         "stream": "f32", "shifted": True, "layers": 1, "sublayers": 1, "cin": 138, "cout": 69, "ape": False,
         "members_t": False, "sampler_steps": 10, "forecast_steps": 1}
    c.update(kw)
    return c


def listed():
    return [
        # The smallest call: one shifted un-modulated block on a 32 x 64 grid (the benchmark's first configuration).  Eight
        # launches of a few microseconds each: what a user sees here is launch and host time.
        _case("block", "block_32x64", 32, 64, 8, 8, 128, 4, 32, 512, "spec", mod_ways=0, stream="bf16"),
        # The second configuration: 1-degree grid, 12 x 12 windows, bf16 stream.  A kernel is a few rounds of workgroups.
        _case("block", "block_180x360", 180, 360, 12, 12, 512, 8, 64, 2048, "spec", mod_ways=0, stream="bf16"),
        # The third: one block on the full quarter-degree grid.
        _case("block", "block_720x1440", 720, 1440, 16, 16, 1024, 16, 64, 4096, "spec", mod_ways=2),
        # The reference's block form at an odd size: rectangular windows, head_dim 128, two members with a noise level
        # each, token and channel counts that are no multiple of a GEMM tile.
        _case("block", "block_ref_ragged", 60, 104, 12, 8, 384, 3, 128, 1088, "ref", batch=2, members_t=True),
        # The denoiser of the benchmark (24 blocks, dim 1536) on a coarse grid: the shape of regional runs, of
        # low-resolution studies and of this repository's depth tests.
        _case("denoiser", "denoiser_64x128", 64, 128, 16, 16, 1536, 24, 64, 6144, "spec", layers=24),
        # ... and on the full 720 x 1440 grid: the headline workload.
        _case("denoiser", "denoiser_720x1440", 720, 1440, 16, 16, 1536, 24, 64, 6144, "spec", layers=24),
        # The reference's science model (8 layers x 3 sublayers, 12 heads x 128, 60 x 60 windows, positional encoding,
        # 144 -> 70 channels) on a coarse grid of four windows.
        _case("denoiser", "denoiser_ref_120x120", 120, 120, 60, 60, 1536, 12, 128, 6144, "ref", layers=8, sublayers=3,
              cin=144, cout=70, ape=True),
        # ... and six of its blocks on the full grid (72 windows of 3600 tokens).
        _case("denoiser", "denoiser_ref_720x1440", 720, 1440, 60, 60, 1536, 12, 128, 6144, "ref", layers=6, cin=144,
              cout=70, ape=True),
        # A narrow model on a 2-degree-class grid: three members as batch with a noise level each, dim 320 = 5 heads x 64,
        # 12 x 12 windows, bf16 stream.
        _case("denoiser", "denoiser_ens_96x180", 96, 180, 12, 12, 320, 5, 64, 1280, "spec", layers=6, batch=3,
              members_t=True, stream="bf16", mod_ways=3),
        # One eager draw of the 10-step sampler with a small model: 19 denoiser calls in a row, host-bound.
        _case("sample", "sample_32x64", 32, 64, 16, 16, 256, 4, 64, 1024, "ref", layers=4),
        # Two ensemble forecast steps on the 1-degree grid, one HIP graph per step: 4 members, forcings, conditioning and
        # feedback on the device, 38 denoiser calls.
        _case("forecast", "forecast_180x360", 180, 360, 12, 12, 512, 8, 64, 2048, "spec", layers=2, batch=4,
              cin=144, forecast_steps=2),
    ]


# ----------------------------------------------------------------------------------------------
# drawn cases

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block"] * 5 + ["denoiser"] * 4 + ["sample"])
    preset = rng.choice(["spec", "spec", "ref"])
    if preset == "spec":  # bias table and mask: square windows, head_dim 64 or (narrow models) 32
        ws_y = ws_x = rng.choice([8, 12, 16, 16])
        head_dim = rng.choice([32, 64, 64, 64])
    else:  # any window of up to 4096 tokens
        ws_y, ws_x = (_log_int(rng, 6, 60) for _ in range(2))
        head_dim = rng.choice([64, 128])
    width = _log_int(rng, 128, 1536)
    dim = max(128, width // 64 * 64)
    if dim % head_dim:
        dim += 64
    heads = dim // head_dim
    mlp = dim * rng.choice([2, 3, 4, 4]) + 64 * rng.randrange(0, 3)
    tokens = _log_int(rng, 2048, 1036800 if kind != "sample" else 65536)
    batch = rng.choice([1, 1, 1, 2, 3, 4])
    tokens = max(2048, tokens // batch)
    windows = max(2, int(round(tokens / (ws_y * ws_x))))
    ny = max(1, int(round(math.sqrt(windows * ws_x / (2.0 * ws_y)))))
    nx = max(1, int(round(windows / ny)))
    ways = 3 if preset == "ref" else rng.choice([0, 2, 2, 3]) if kind == "block" else rng.choice([2, 3])
    case = _case(kind, "", ny * ws_y, nx * ws_x, ws_y, ws_x, dim, heads, head_dim, mlp, preset, batch=batch,
                 mod_ways=ways, stream=rng.choice(["f32", "f32", "bf16"]), shifted=rng.random() < 0.5,
                 members_t=batch > 1 and rng.random() < 0.5 and kind != "sample",
                 layers=rng.randint(1, 24) if kind == "denoiser" else rng.randint(1, 6) if kind == "sample" else 1,
                 cout=rng.randint(4, 80), ape=kind == "denoiser" and rng.random() < 0.5,
                 sampler_steps=rng.randint(2, 10))
    # state channels and conditioning (an equal number of channels, and forcings)
    case["cin"] = min(159, 2 * case["cout"] + rng.randint(0, 12)) if kind != "block" else 138
    if kind == "denoiser":
        case["cin"] = max(8, case["cin"])
    while case["layers"] > 1 and work(case)["flops"] > MAX_DRAW_FLOPS:
        case["layers"] -= 1
    while case["sampler_steps"] > 2 and work(case)["flops"] > MAX_DRAW_FLOPS:
        case["sampler_steps"] -= 1
    del case["name"]
    return case


# ----------------------------------------------------------------------------------------------
# one pass

def _options(case):
    if case["preset"] == "ref":
        return dict(preset="ref")
    return dict(preset="spec", mod_ways=case["mod_ways"])


def _fill(module, g):
    """Unit-gain random weights, norm gains around 1, small biases, modulation around the identity."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            r = torch.randn(p.shape, generator=g, device=p.device, dtype=torch.float32)
            if name.endswith("relative_position_bias_table"):
                r *= 0.5
            elif "modulation.2.weight" in name:  # shift, scale and gate vectors of a few tenths
                r *= 0.3 * p.shape[1] ** -0.5
            elif p.dim() >= 2:
                r *= p.shape[1] ** -0.5
            else:
                r *= 0.1
                if name.endswith("weight"):
                    r += 1.0
            p.copy_(r.to(p.dtype))
            if "modulelist" in name and name.endswith("modulation.2.bias") and module.opts.mod_ways == 3:
                d = p.numel() // 6
                p[2 * d:3 * d] += 1.0  # gates around 1
                p[5 * d:] += 1.0


def _model(case, g):
    with torch.device(DEVICE):
        m = amd.LocalAERIS(device_mesh=None, heads=case["heads"], dim=case["dim"], head_dim=case["head_dim"],
                           mlp_dim=case["mlp"], window_size=(case["ws_y"], case["ws_x"]),
                           image_shape=(case["H"], case["W"]), rope_base=10_000, sublayers=case["sublayers"],
                           sinusoidal_emb_max_period=10_000, n_layers=case["layers"] + 2, model_in_channels=case["cin"],
                           model_out_channels=case["cout"],
                           residual_dtype=torch.bfloat16 if case["stream"] == "bf16" else torch.float32, **_options(case))
    _fill(m, g)
    if case["ape"]:
        m.generate_ape(DEVICE)
    return m


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    B, S, d, C = case["batch"], case["H"] * case["W"], case["dim"], case["cout"]
    kind = case["kind"]

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEVICE)

    if kind == "block":
        with torch.device(DEVICE):
            layer = amd.SwinLayer(None, d, case["heads"], case["head_dim"], case["mlp"], (case["ws_y"], case["ws_x"]),
                                  (case["H"], case["W"]), case["shifted"], 10_000, **_options(case)).to(torch.bfloat16)
        _fill(layer, g)
        x = randn(B, S, d).to(torch.bfloat16 if case["stream"] == "bf16" else torch.float32)
        t = randn(B if case["members_t"] else 1, d) if case["mod_ways"] else None
        # preset "ref" does not shift on its own: the caller passes the shift of the odd layers
        shift = (case["ws_y"] // 2, case["ws_x"] // 2) if case["shifted"] else (0, 0)
        return {"kind": kind, "layer": layer, "x": x, "t": t, "shift": shift}
    model = _model(case, g)
    if kind == "denoiser":
        t = torch.rand(B if case["members_t"] else 1, generator=g, device=DEVICE) * (math.pi / 2)
        return {"kind": kind, "model": model, "x": randn(B, S, case["cin"]), "t": t}
    sampler = amd.TrigFlowSampler(model, n_steps=case["sampler_steps"], device=DEVICE)
    if kind == "sample":
        return {"kind": kind, "sampler": sampler, "cond": randn(B, S, case["cin"] - C), "latents": randn(B, S, C)}
    n = case["forecast_steps"]
    forcing = (case["cin"] - 2 * C) // 2
    ro = sampler.begin_rollout(randn(B, S, C), n, x_mean=randn(C), x_std=0.5 + torch.rand(C, generator=g, device=DEVICE),
                               t_mean=0.1 * randn(C), t_std=0.2 + 0.2 * torch.rand(C, generator=g, device=DEVICE),
                               forcing=randn(n + 1, 1, S, forcing) if forcing else None, latents=randn(n, B, S, C),
                               use_graph=True, graph_warmup=1)
    return {"kind": kind, "rollout": ro}


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "block":
        return state["layer"](state["x"], state["t"], shift=state["shift"])
    if kind == "denoiser":
        return state["model"](state["x"], state["t"])
    if kind == "sample":
        return state["sampler"].sample(state["cond"], state["latents"])
    ro = state["rollout"]
    ro.reset()
    return ro.run()


# ----------------------------------------------------------------------------------------------
# what one pass cannot do without

def _blocks(case):
    return case["layers"] * case["sublayers"]


def _block_work(case):
    """FLOP and weight bytes of one block on the case's batch."""
    T, d, hid = case["batch"] * case["H"] * case["W"], case["dim"], case["mlp"]
    inner, ref = case["heads"] * case["head_dim"], case["preset"] == "ref"
    mats = d * 3 * inner + inner * d + d * hid * (3 if ref else 2)
    mod = d * d + d * 2 * case["mod_ways"] * d if case["mod_ways"] else 0
    rows = case["batch"] if case["members_t"] else 1
    flops = 2.0 * T * mats + 4.0 * T * case["ws_y"] * case["ws_x"] * inner + 2.0 * rows * mod
    return flops, 2.0 * mats + 4.0 * mod


def work(case):
    T, d = case["batch"] * case["H"] * case["W"], case["dim"]
    flops, weights = _block_work(case)
    if case["kind"] == "block":
        return {"bytes": 2.0 * T * d * (2 if case["stream"] == "bf16" else 4) + weights, "flops": flops}
    n = _blocks(case)
    ends = case["cin"] * d + 3 * d * d + d * case["cout"]
    one_flops = n * flops + 2.0 * T * d * (case["cin"] + case["cout"])
    # the weights count once per call: a denoiser's 24 blocks do not stay on the chip from one call to the next
    one_bytes = n * weights + 4.0 * ends + 4.0 * T * (case["cin"] + case["cout"])
    if case["ape"]:
        one_bytes += 4.0 * case["H"] * case["W"] * case["cin"]
    calls = 1
    if case["kind"] in ("sample", "forecast"):
        calls = (2 * case["sampler_steps"] - 1) * case["forecast_steps"]
    return {"bytes": calls * one_bytes, "flops": calls * one_flops}


def tolerance(case):
    """Relative 2-norm error another correct implementation at this precision may show: about four times the distance to
    an fp32 evaluation with the same weights.  Measured: blocks 1.8e-3 (f32 stream) and 2.9e-3 .. 3.1e-3 (bf16 stream, whose
    result is rounded), a 24-block denoiser with an f32 stream 2.5e-3, a 10-step draw 1.1e-3, a six-block denoiser with
    a bf16 stream 5.8e-3 (two roundings of the stream per block, adding up with depth)."""
    if case["stream"] == "f32":
        return {"rel": 1.0e-2}
    return {"rel": 1.2e-2 if case["kind"] == "block" else 2.4e-2}
