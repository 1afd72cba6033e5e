"""Performance cases of the attention path and of the models around it.

Each case is one call that a program using this package makes over and over: an
attention operator call (sampling, forward + tangent, training), a model forward +
tangent, a training step, a sampling loop.  ``listed()`` gives a fixed set,
``draw()`` further ones of the same ranges, ``prepare`` / ``run`` build and execute a
case on the current GPU, ``work`` states its algorithmic bytes and operations and
``tolerance`` how far two correct implementations may differ.
"""
from __future__ import annotations

import contextlib
import math

import torch
import torch.autograd.forward_ad as fwAD

from dmf_amd import flash_attn_func, flash_attn_qknorm_qkvpacked_func, flash_attn_qkvpacked_func
from dmf_amd.dmft import DMFT
from dmf_amd.harness import GraphedStep, meanflow_jvp, synthetic_batch, train_step
from dmf_amd.layers import frozen_low_precision_params
from dmf_amd.samplers import euler_sampler

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _attn(name, layout, mode, dtype, B, H, N, D):
    return {"name": name, "kind": "attn", "layout": layout, "mode": mode, "dtype": dtype, "B": B, "H": H, "N": N, "D": D}


def _model(name, mode, B, grid, hidden, heads, depth, dmf_depth, qk_norm=False, graph=False):
    return {"name": name, "kind": "model", "mode": mode, "B": B, "grid": grid, "hidden": hidden, "heads": heads,
            "depth": depth, "dmf_depth": dmf_depth, "qk_norm": qk_norm, "graph": graph}


def listed():
    return [
        # one layer's attention while ONE image is sampled with guidance (a batch of two): the latency end
        _attn("infer_b2_n256", "packed", "infer", "bf16", 2, 16, 256, 72),
        # sampling in half precision at 512 px (the samplers' fp16 option): operator on views of the packed projection
        _attn("infer_fp16_n1024", "views", "infer", "fp16", 8, 16, 1024, 72),
        # forward + tangent at the XL/2 512 px shape, the operator call of the MeanFlow target at a large batch
        _attn("jvp_xl2_n1024", "separate", "jvp", "bf16", 64, 16, 1024, 72),
        # the same call of the B/2 model at 256 px, on the packed projection output
        _attn("jvp_b2_n256", "packed", "jvp", "bf16", 64, 12, 256, 64),
        # one layer of the XL/2 256 px training step: forward + tangent, backward on the primal output
        _attn("train_xl2_n256", "packed", "jvp_train", "bf16", 32, 16, 256, 72),
        # one layer of the XL/2 512 px training step, q and k RMS-normalised inside the operator
        _attn("train_xl2_n1024_qknorm", "qknorm", "jvp_train", "bf16", 16, 16, 1024, 72),
        # flow-matching training (forward + backward, no tangent) on a token count that is a multiple of nothing
        _attn("train_ragged_n333", "separate", "train", "bf16", 6, 12, 333, 64),
        # training in full precision
        _attn("train_fp32_n256", "separate", "jvp_train", "fp32", 16, 12, 256, 64),
        # long sequence at the largest head dim
        _attn("train_n2048_d128", "separate", "jvp_train", "bf16", 2, 16, 2048, 128),
        # DMFT-B/2 at 256 px, whole-model forward + tangent under autocast, replayed as a captured step
        _model("dmft_b2_jvp", "jvp", 64, 16, 768, 12, 12, 8, graph=True),
        # DMFT-XL/2 training step at 256 px, batch 32 (MeanFlow loss: forward + tangent, backward), launched eagerly; four
        # blocks at the full width stand for the twenty-eight
        _model("dmft_xl2x4_train", "train", 32, 16, 1152, 16, 4, 3),
        # generation: DMFT-B/2 in bf16, eight images, four steps with classifier-free guidance
        _model("dmft_b2_sample", "sample", 8, 16, 768, 12, 12, 8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.75:
        dtype = rng.choice(["bf16"] * 6 + ["fp32", "fp16"])
        layout = rng.choice(["separate", "views"] if dtype == "fp16" else ["separate", "views", "packed", "packed", "qknorm"])
        mode = rng.choice(["infer", "jvp", "train", "jvp_train"])
        H, D = rng.choice([(6, 64), (12, 64), (16, 64), (16, 64), (16, 72), (16, 72), (16, 72), (16, 72), (16, 80), (16, 128)])
        N = rng.choice([256, 1024, _log_int(rng, 16, 2048), _log_int(rng, 16, 2048), _log_int(rng, 64, 1024)])
        # at most the work of the largest listed case of the kind (and, for the slower types, of its time)
        most = 9e11 if dtype == "bf16" else 6e10
        units = {"infer": 4, "jvp": 12, "train": 14, "jvp_train": 22}[mode]
        B = _log_int(rng, 1, max(1, min(64, int(most / (units * H * N * N * D)))))
        case = _attn("", layout, mode, dtype, B, H, N, D)
    else:
        mode = rng.choice(["jvp", "train", "sample"])
        hidden, heads = rng.choice([(384, 6), (768, 12), (1024, 16), (1152, 16)])
        grid = rng.choice([8, 16, 16, rng.randint(4, 20), 32])
        depth = rng.randint(2, 4)
        B = _log_int(rng, 1, max(1, min(64, 32 * 256 // (grid * grid))))
        case = _model("", mode, B, grid, hidden, heads, depth, rng.randint(1, depth - 1), rng.random() < 0.4,
                      mode == "jvp" and rng.random() < 0.5)
    del case["name"]
    return case


# ---- attention operator ----------------------------------------------------------------------------------------------

def _prepare_attn(case, gen, device):
    B, N, H, D, dt = case["B"], case["N"], case["H"], case["D"], DTYPES[case["dtype"]]
    dual, train = "jvp" in case["mode"], "train" in case["mode"]
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=device, dtype=torch.float32)
    st = {"kind": "attn", "layout": case["layout"], "mode": case["mode"], "dual": dual, "train": train}
    if case["layout"] in ("packed", "qknorm", "views"):
        prim = [rand(B, N, 3, H, D).to(dt)]
        tang = [rand(B, N, 3, H, D).to(dt)] if dual else []
        if case["layout"] == "views":      # q, k, v as slices of the projection output
            prim = list(prim[0].unbind(2))
            tang = list(tang[0].unbind(2)) if dual else []
    else:
        prim = [rand(B, N, H, D).to(dt) for _ in range(3)]
        tang = [rand(B, N, H, D).to(dt) for _ in range(3)] if dual else []
    st["prim"] = [p.requires_grad_(train) for p in prim]
    st["tang"] = tang
    if case["layout"] == "qknorm":
        st["gains"] = [(1 + 0.1 * rand(D)).requires_grad_(train) for _ in range(2)]
    if train:
        st["dout"] = rand(B, N, H, D).to(dt)
    return st


def _call_attn(st, args):
    if st["layout"] == "packed":
        return flash_attn_qkvpacked_func(*args)
    if st["layout"] == "qknorm":
        return flash_attn_qknorm_qkvpacked_func(*args, *st["gains"])
    return flash_attn_func(*args)


def _run_attn(st):
    if not st["train"]:
        if st["dual"]:
            return torch.func.jvp(lambda *a: _call_attn(st, a), tuple(st["prim"]), tuple(st["tang"]))
        with torch.no_grad():
            return _call_attn(st, st["prim"])
    leaves = st["prim"] + st.get("gains", [])
    if not st["dual"]:
        out = _call_attn(st, st["prim"])
        return out.detach(), torch.autograd.grad(out, leaves, st["dout"])
    with fwAD.dual_level():
        out, tout = fwAD.unpack_dual(_call_attn(st, [fwAD.make_dual(p, t) for p, t in zip(st["prim"], st["tang"])]))
    return out.detach(), tout.detach(), torch.autograd.grad(out, leaves, st["dout"])


def _work_attn(case):
    B, N, H, D = case["B"], case["N"], case["H"], case["D"]
    dual, train = "jvp" in case["mode"], "train" in case["mode"]
    elem = B * N * H * D
    tensors = 4 * (2 if dual else 1) + (4 if train else 0)      # q k v o, their tangents; dout and three gradients
    gemms = (6 if dual else 2) + (5 if train else 0)            # score-sized products of 2 B H N^2 D operations
    return {"bytes": tensors * elem * torch.finfo(DTYPES[case["dtype"]]).bits // 8, "flops": gemms * 2 * B * H * N * N * D}


# ---- models ------------------------------------------------------------------------------------------------------------

def _prepare_model(case, seed, device):
    size = 2 * case["grid"]
    with torch.device(device):
        model = DMFT(input_size=size, patch_size=2, hidden_size=case["hidden"], depth=case["depth"], num_heads=case["heads"],
                     dmf_depth=case["dmf_depth"], qk_norm=case["qk_norm"], attn_func="hip", block_ops="hip")
    model.init_trunc_normal_(0.02, seed)
    st = {"kind": "model", "mode": case["mode"], "model": model}
    if case["mode"] == "train":
        st["data"] = synthetic_batch(case["B"], device, seed=seed, input_size=size)
        st["params"] = [p for p in model.parameters() if p.requires_grad]
    elif case["mode"] == "jvp":
        st["data"] = synthetic_batch(case["B"], device, seed=seed, input_size=size)
        model.requires_grad_(False)
        # weights are frozen for as long as the state lives: one low-precision copy, as the evaluation loop makes it
        st["frozen"] = contextlib.ExitStack()
        st["frozen"].enter_context(frozen_low_precision_params(model))

        def step(*batch):
            with torch.autocast("cuda", dtype=torch.bfloat16):
                return meanflow_jvp(model, *batch)
        st["step"] = GraphedStep(step, *st["data"]) if case["graph"] else step
    else:
        st["model"] = model.to(torch.bfloat16).eval().requires_grad_(False)
        z, _, _, y, _ = synthetic_batch(case["B"], device, seed=seed, input_size=size)
        st["data"] = (z.to(torch.bfloat16), y)
    return st


def _run_model(st):
    if st["mode"] == "jvp":
        return st["step"](*st["data"])
    if st["mode"] == "sample":
        return euler_sampler(st["model"], *st["data"], num_steps=4, cfg_scale=1.5, g_min=0.0, g_max=0.8)
    st["model"].zero_grad(set_to_none=True)
    loss = train_step(st["model"], st["data"])
    return loss.detach(), [p.grad for p in st["params"]]


def _work_model(case):
    B, N, C, depth = case["B"], case["grid"] ** 2, case["hidden"], case["depth"]
    # multiply-adds of one forward on B images: blocks (qkv, proj, MLP; attention), their modulation, patch embedding + output
    macs = B * (depth * (12 * N * C * C + 2 * N * N * C + 6 * C * C) + 2 * C * C + 32 * N * C)
    # attention with tangents takes three times the primal products (and 2.5 times in the backward), a linear layer twice
    attn = 2 * B * depth * N * N * C
    params = depth * 18 * C * C + 2 * C * C + 32 * C + 1001 * C
    image = B * 4 * (2 * case["grid"]) ** 2
    if case["mode"] == "jvp":
        return {"bytes": 2 * params + 4 * 4 * image, "flops": 2 * (2 * macs + attn)}
    if case["mode"] == "sample":     # guided on t <= 0.8 of the knots 1, 0.75, 0.5, 0.25: 1 + 2 + 2 + 2 forwards on B images
        return {"bytes": 2 * params + 10 * image, "flops": 2 * 7 * macs}
    # training: forward + tangent, then the backward (two products per linear layer, five for the attention's two)
    return {"bytes": 8 * params + 2 * 4 * image, "flops": 2 * (2 * macs + attn + 2 * macs + attn // 4)}


# ---- interface ---------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] == "model":
        return _prepare_model(case, seed, device)
    return _prepare_attn(case, torch.Generator(device=device).manual_seed(seed), device)


def run(state):
    return _run_model(state) if state["kind"] == "model" else _run_attn(state)


def work(case):
    return _work_model(case) if case["kind"] == "model" else _work_attn(case)


def tolerance(case):
    # About four times the distance to the same path evaluated in 64 bits (attention) or in fp32 by library operators (models),
    # worst output of the listed and some thirty drawn cases: bf16 3.2e-3, with the q / k norms in front up to 5.7e-3; fp16
    # 2.1e-4 (its output rounding); fp32 9.3e-7; models 4e-3 to 9e-3, the largest in small gradients of deep small models.
    if case["kind"] == "model":
        return {"rel": 2.5e-2}
    if case["layout"] == "qknorm" and case["dtype"] == "bf16":
        return {"rel": 2e-2}
    return {"bf16": {"rel": 1.2e-2}, "fp16": {"rel": 8e-4}, "fp32": {"rel": 4e-6}}[case["dtype"]]
