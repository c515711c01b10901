"""The workloads whose speed is measured: VMonarch attention and flash-entropy attention, forward alone
(inference) and forward + backward (training), called as a diffusion-transformer program calls them.

A case is a dict of plain values:
  op      "fea" (flash_entropy_attention) or "vmonarch" (VMonarchAttention)
  train   False: the forward under no_grad; True: forward and gradients of q, k, v
  B, H, D, Dv, dtype
  layout  "bhnd": contiguous (B, H, N, D) tensors; "bnhd": (B, N, H, D) buffers viewed as (B, H, N, D), the
          memory order of a transformer block's projections
  N       tokens ("fea");  m, b, iters, rt: grid rows, tokens per grid row, alternating-minimisation steps,
          recomputed leading tokens ("vmonarch", N = m * b)
"""
import math

import torch

from vmonarch_amd import VMonarchAttention, flash_entropy_attention

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _fea(name, B, H, N, D, Dv, dtype="bf16", train=False, layout="bhnd"):
    return {"name": name, "op": "fea", "train": train, "B": B, "H": H, "N": N, "D": D, "Dv": Dv, "dtype": dtype,
            "layout": layout}


def _vmonarch(name, B, H, m, b, D, dtype="bf16", iters=2, rt=0, train=False, layout="bhnd"):
    return {"name": name, "op": "vmonarch", "train": train, "B": B, "H": H, "m": m, "b": b, "D": D, "Dv": D,
            "dtype": dtype, "iters": iters, "rt": rt, "layout": layout}


def listed():
    return [
        # one short sequence, two heads: a single small call, where latency counts
        _fea("fea_fwd_short", 1, 2, 1024, 64, 64),
        # an ordinary batch of image-sized sequences
        _fea("fea_fwd_image", 2, 4, 4096, 128, 128),
        # row blocks with values twice as wide as the heads ([k | v], as the row-block seam calls it), odd length
        _fea("fea_fwd_wide_values", 1, 48, 777, 64, 128, dtype="f16", layout="bnhd"),
        # training on an odd, short sequence
        _fea("fea_train_odd", 2, 4, 1000, 64, 64, dtype="f16", train=True),
        # training on a long sequence: the largest case
        _fea("fea_train_long", 1, 24, 16384, 128, 128, train=True),
        # the smallest VMonarch call: a toy grid of four rows
        _vmonarch("vmonarch_fwd_toy", 1, 2, 4, 64, 64, dtype="f16", rt=64),
        # a small grid, batch of two (e.g. a low-resolution clip with guidance)
        _vmonarch("vmonarch_fwd_clip", 2, 4, 16, 256, 128, rt=256),
        # the video workload: 21 latent frames of 1560 tokens, first frame exact
        _vmonarch("vmonarch_fwd_video", 1, 12, 21, 1560, 128, rt=1560),
        # ... and its training step, on a transformer block's own buffers
        _vmonarch("vmonarch_train_video", 1, 12, 21, 1560, 128, rt=1560, train=True, layout="bnhd"),
        # 33 latent frames (129 video frames) of an odd frame size
        _vmonarch("vmonarch_fwd_33_frames", 1, 12, 33, 993, 128, rt=993, layout="bnhd"),
        # training on an odd small grid, narrower heads, three steps, no exact rows
        _vmonarch("vmonarch_train_odd", 1, 8, 48, 211, 64, dtype="f16", iters=3, train=True),
        # training on a long clip: many frames, small ones
        _vmonarch("vmonarch_train_96_frames", 1, 12, 96, 341, 128, rt=341, train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MAX_DRAWN_FLOPS = 3.0e12   # a quarter of the largest listed case's


def draw(rng):
    while True:
        D = rng.choice([64, 128])
        common = {"train": rng.random() < 0.5, "B": rng.choice([1, 1, 2]), "D": D,
                  "dtype": rng.choice(["bf16", "bf16", "f16"]), "layout": rng.choice(["bhnd", "bnhd"])}
        if rng.random() < 0.4:
            case = {"op": "fea", "H": _log_int(rng, 1, 48), "N": _log_int(rng, 128, 16384),
                    "Dv": rng.choice([D, D, 2 * D]), **common}
        else:
            m, b = _log_int(rng, 4, 128), _log_int(rng, 32, 2048)
            case = {"op": "vmonarch", "H": _log_int(rng, 2, 24), "m": m, "b": b, "Dv": D,
                    "iters": rng.choice([1, 2, 2, 3]), "rt": rng.choice([0, b]), **common}
            if m * b > 33000:
                continue
        if work(case)["flops"] <= _MAX_DRAWN_FLOPS:
            return case


def _tokens(case):
    return case["N"] if case["op"] == "fea" else case["m"] * case["b"]


def _inputs(case, seed):
    """q, k, v (and for training the upstream gradients) from the seed alone: unit normal q, k, v for the plain
    attention; q, k of half that (the soft logits of a normalised video transformer) for VMonarch."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    B, H, N, dt = case["B"], case["H"], _tokens(case), DTYPES[case["dtype"]]

    def tensor(feat, scale=1.0):
        shape = (B, H, N, feat) if case["layout"] == "bhnd" else (B, N, H, feat)
        t = torch.randn(shape, generator=g, device=dev).mul_(scale).to(dt)
        return t if case["layout"] == "bhnd" else t.transpose(1, 2)

    qk = 1.0 if case["op"] == "fea" else 0.5
    out = {"q": tensor(case["D"], qk), "k": tensor(case["D"], qk), "v": tensor(case["Dv"])}
    if case["train"]:
        out["dout"] = tensor(case["Dv"])
        if case["op"] == "fea":
            out["dent"] = torch.randn((B, H, N), generator=g, device=dev)
    return out


def prepare(case, seed):
    state = _inputs(case, seed)
    if case["train"]:
        for name in "qkv":
            state[name].requires_grad_()
    if case["op"] == "vmonarch":
        state["attn"] = VMonarchAttention(case["m"], case["b"], num_iters=case["iters"])
        state["rt"] = case["rt"]
    return state


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    train = "dout" in state
    with torch.set_grad_enabled(train):
        if "attn" in state:
            outs = (state["attn"](q, k, v, recompute_tokens=state["rt"]),)
        else:
            outs = flash_entropy_attention(q, k, v)
    if not train:
        return list(outs)
    upstream = (state["dout"],) if len(outs) == 1 else (state["dout"], state["dent"])
    grads = torch.autograd.grad(outs, (q, k, v), upstream)
    return [t.detach() for t in outs] + list(grads)


def work(case):
    B, H, N, D, Dv = case["B"], case["H"], _tokens(case), case["D"], case["Dv"]
    tok = B * H * N
    nbytes = tok * (2 * D + 2 * Dv) * 2          # q, k, v read; o / z written
    if case["op"] == "fea":
        flops = 2.0 * tok * N * (D + Dv)
        nbytes += tok * 4                        # the entropies
    else:
        m, b, it, rt = case["m"], case["b"], case["iters"], min(case["rt"], N)
        flops = 2.0 * tok * b * (2 * D * it + Dv)          # R-steps: values k, the last one [k | v]
        flops += 2.0 * tok * m * (2 * D * (it - 1) + D + Dv)   # L-steps
        flops += 2.0 * B * H * rt * N * (D + Dv)           # the exact rows
    if case["train"]:
        flops *= 3.5                             # the backward has five products for the forward's two
        nbytes += tok * (2 * D + 2 * Dv) * 2     # the upstream gradient read; dq, dk, dv written
        nbytes += tok * 4 if case["op"] == "fea" else 0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times what the outputs were seen off `exact` by, over the listed cases and thirty drawn ones: 2.4e-3 (bf16)
    and 3.0e-4 (fp16) for the plain attention, whose results are rounded once, 4.6e-3 and 5.5e-4 for VMonarch,
    which stores u and the row outputs in 16 bits between its steps; the largest single difference 5.1e-2 and
    3.4e-3 of the result's root mean square."""
    bf16 = case["dtype"] == "bf16"
    rel = (1e-2 if bf16 else 1.2e-3) if case["op"] == "fea" else (1.8e-2 if bf16 else 2.2e-3)
    return {"rel": rel, "max": 0.2 if bf16 else 1.4e-2}


def _exact_fea(q, k, v, scale):
    """Attention and row entropies of one head, any number of leading dims."""
    s = q @ k.transpose(-1, -2) * scale
    logp = torch.log_softmax(s, -1)
    p = logp.exp()
    return p @ v, -(p * logp).sum(-1)


def _exact_vmonarch(q, k, v, m, b, iters, rt, min_col_mass=0.01):
    """VMonarch attention of one head: (N, D) tensors."""
    scale = q.shape[-1] ** -0.5
    qg, kg, vg = (t.view(m, b, -1) for t in (q, k, v))
    u, y = qg * scale, None
    for it in range(iters):
        s = u @ kg.transpose(-1, -2)
        logp = torch.log_softmax(s, -1)
        p = logp.exp()
        ent = -(p * logp).sum(-1).detach()                     # (m, b)
        kr = p @ kg * scale
        logits = qg.transpose(0, 1) @ kr.permute(1, 2, 0)      # (b, m, m): query row i, key row j of a column
        attn = torch.softmax(logits + ent.transpose(0, 1).unsqueeze(1), -1)
        if it == iters - 1:
            y = (attn @ (p @ vg).transpose(0, 1)).transpose(0, 1)
        else:
            mass = attn.sum(1).clamp_min(min_col_mass)         # (b, m)
            u = (attn.transpose(1, 2) @ qg.transpose(0, 1) * (scale / mass).unsqueeze(-1)).transpose(0, 1)
    z = y.reshape(m * b, -1)
    if rt > 0:
        z = torch.cat([torch.softmax(q[:rt] @ k.transpose(0, 1) * scale, -1) @ v, z[rt:]], 0)
    return z


def exact(case, seed):
    x = _inputs(case, seed)
    B, H, N = case["B"], case["H"], _tokens(case)
    results = []
    for bi in range(B):
        for h in range(H):
            q, k, v = (x[n][bi, h].double() for n in "qkv")
            if case["train"]:
                q, k, v = (t.requires_grad_() for t in (q, k, v))
            with torch.set_grad_enabled(case["train"]):
                if case["op"] == "fea":
                    outs = _exact_fea(q, k, v, case["D"] ** -0.5)
                else:
                    outs = (_exact_vmonarch(q, k, v, case["m"], case["b"], case["iters"], min(case["rt"], N)),)
            if case["train"]:
                upstream = [x["dout"][bi, h].double()] + ([x["dent"][bi, h].double()] if len(outs) > 1 else [])
                outs = [t.detach() for t in outs] + list(torch.autograd.grad(outs, (q, k, v), upstream))
            results.append(outs)
    return [torch.stack(parts).view(B, H, *parts[0].shape) for parts in zip(*results)]
