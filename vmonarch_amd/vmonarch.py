"""
VMonarch attention (drop-in for video_monarch_attention/vmonarch.py of the reference).

The N = m * b tokens are laid out on an (m, b) grid, token n -> (n // b, n % b).  The attention
map is approximated by a Monarch matrix built from
  - R: m dense (b x b) blocks, mixing tokens inside each grid row (a batched flash-entropy
    attention, the R-step);
  - L: b dense (m x m) blocks, mixing tokens inside each grid column (the L-step);
fitted by a few steps of alternating minimisation (reference: vmonarch.py:1-11, :29-69).

Execution paths, with identical results within bf16 tolerance:
  * fused (forward without autograd): every step is a gfx950 HIP kernel -- the R-step reads the
    (B, H, m*b, D) tensors in place as m frames per head (no flatten copy, no torch.cat of
    [k | v]), the L-step is one fused kernel per iteration (one MFMA tile per grid column for
    m <= 32, a general kernel beyond), and the recompute of the first tokens is a split-KV flash
    kernel writing straight into z;
  * _VMonarchFunction (autograd): the same forward keeping its activations, and a HIP backward;
  * head-dim mixes the kernels do not take as they are (16 with 32; D != Dv with autograd; neither
    is a shape the reference's VMonarch runs) run either of the above on q, k, v zero-padded to one
    kernel width;
  * composed: the reference's structure step by step (R-step through the `_row_block_attention`
    seam, L-step as torch tensor ops), used when a caller replaced `_row_block_attention`
    (tests/test_vmonarch.py:59 does), and -- with a RuntimeWarning -- for shapes no HIP path takes.
"""
import warnings

import torch
import torch.nn as nn

from . import _lib
from .kernel import flash_entropy_attention

# number of CUs on an MI355X; the recompute picks its split-KV count to fill them
_NUM_CUS = 256


def _row_block_attention(x, k, w):
    """Attention inside every grid row (reference vmonarch.py:19-26).

    x, k: (B, H, m, b, D); w: (B, H, m, b, Dw).
    Returns softmax(x k^T) w and sum_j P_ij log P_ij (= -entropy) for every row of P.
    """
    out, ent = flash_entropy_attention(*(t.flatten(1, 2) for t in (x, k, w)), sm_scale=1.0)
    return out.view(*w.shape[:-1], -1), -ent.view(x.shape[:-1]).detach()


_ROW_BLOCK_ATTENTION = _row_block_attention   # the seam as shipped; patched seams use the composed path


def _recompute_splits(problems, nq, nk, paired=False):
    """Key splits of the recompute, each merged from fp32 partials by one more launch.

    On its own: the fewest that fill ~80% of one round of workgroup slots (two 128-query workgroups per CU), each
    split keeping >= 512 keys (measured at cfg4, 156 query tiles: 3 splits 0.300 ms, 8 splits 0.309, 16 splits 0.336).
    In one launch with R-step 0, whose workgroups fill the other slots: the fewest that make 120 workgroups, at least
    two (one workgroup walking all keys would outlast the R-step) until the recompute's tiles fill a round by themselves
    (the line of the rule above, 409 tiles; from there a second split only writes and merges partials), and at most
    eight, each of >= 256 keys.  Measured, whole forward in us at 2 / 4 / 8 / 16 splits: 16 query tiles x 4096 keys
    75.9 / 64.6 / 61.0 / 65.4; 24 x 4200 88.2 / 76.1 / 81.9 / 85.1; 48 x 13200 279 / 255 / 261 / 271; 156 x 32760
    1209 / 1215 / 1237 / 1269.  At 1 / 2 splits: 156 x 32760 1190 / 1153; 252 x 32760 1301 / 1313; 312 x 32760 1441 /
    1429; 624 x 32760 4530 / 4557; 732 x 32760 2164 / 2193; 3072 x 32760 (all tokens) 6277 / 6420, and 406 MB of
    partials."""
    base = problems * ((nq + 127) // 128)
    want = -(-int(0.8 * 2 * _NUM_CUS) // base)
    if paired:
        return max(1, min(8, max(min(2, want), -(-120 // base)), nk // 256))
    return max(1, min(16, want, nk // 512))


def _recompute_plan(B, H, N, D, Dv, num_iters, rt, qk_fp8=False):
    """(order, key splits) of the exact recompute of the first rt queries; see _RECOMPUTE_OVERLAP."""
    order = _RECOMPUTE_OVERLAP
    if rt <= 0:
        return 0, 1
    if order == "auto":
        flops = 2.0 * B * H * rt * N * (D + Dv)
        if num_iters > 1 and D == Dv and (D == 128 or D == 64 and flops < _PAIR_64_MAX_FLOPS) and not qk_fp8:
            order = "with_r0"
        else:
            order = "start" if flops >= _FORK_MIN_FLOPS else "off"
    return _OVERLAPS[order], _recompute_splits(B * H, rt, N, order == "with_r0")


def _lstep_launch(q, out, ent, res, m, b, scale, last, skip, min_col_mass):
    _lib.host().lstep_fwd(q, out, ent, res, m, b, scale, bool(last), skip, min_col_mass)


def _lstep_one_tile(m, d, dv, last):
    """Whether the one-tile L-step kernels take this grid (csrc/lstep.hip one_tile_built)."""
    return m <= 32 and d in (64, 128) and (not last or dv in (64, 128))


def _lstep_bwd_launch(q, out, ent, grad_res, grad_q, grad_out, m, b, scale, last, skip, min_col_mass,
                      overwrite_q=False, delta=None):
    """Backward of one L-step (vmo_lstep_bwd): grad_q (fp32) += dL/dq (= with overwrite_q),
    grad_out = dL/d out; with `delta` ((B, H, N) fp32; one-tile grids, and multi-block ones' last step) also rowsum(out * grad_out)."""
    _lib.host().lstep_bwd(q, out, ent, grad_res, grad_q, grad_out, m, b, scale, bool(last), skip, min_col_mass,
                          bool(overwrite_q), delta)


_LDS_BYTES = 160 * 1024   # per CU on gfx950


def _lstep_general_lds(m, d, dv, last, bwd):
    """LDS bytes per grid column of the general L-step kernels (csrc/lstep.hip lw_layout): 16-bit rows of q,
    kr (and the upstream gradient, y) padded by 16 bytes, one or two fp32 m x (m + 1) matrices, 4 m floats."""
    r16 = lambda b: (b + 15) // 16 * 16   # noqa: E731
    ldq, ldy, ldm = d + 8, dv + 8, m + 1
    total = 2 * r16(m * ldq * 2) + r16(m * ldm * 4) + r16(4 * m * 4)
    if bwd:
        total += r16(m * (ldy if last else ldq) * 2) + r16(m * ldm * 4)
    if last:
        total += r16(m * ldy * 2)
    return total


_MB_MAX_FRAMES = 128
_MB_BWD = True    # the multi-block backward kernels


def _lstep_mb_lds(m, d, dv, last, bwd):
    """LDS bytes per grid column of the multi-block L-step kernels (csrc/lstep_mb.hip mb_layout with whole tiles):
    q and kr tiles (and y, and the upstream gradient) of M = 32 ceil(m / 32) 16-bit rows, M-float vectors, at least
    the four row-store patches.  (The two-block last step up to 40 frames stages compact tiles, which take less:
    this is the bound the host checks.)"""
    M = 32 * ((m + 31) // 32)
    r = lambda b: (b + 255) // 256 * 256   # noqa: E731
    d, dv = max(d, 32), max(dv, 32)   # 16-wide heads sit in 32-wide tiles
    total = 2 * r(M * d * 2) + (r(M * dv * 2) if last else 0) + 2 * r(M * 4) + r(4 * M * 4)
    if bwd:   # the upstream gradient rows, three more vectors, the backward's own row-store patches (half-size
        # ones for the last step up to 64 frames)
        total += r(M * (dv if last else d) * 2) + 3 * r(M * 4) + 4 * (2048 if last and M <= 64 else 4096)
    return max(total, 4 * 4096)


def _lstep_mb(m, d, dv, bwd):
    """Whether the multi-block MFMA L-step kernels take this grid: up to 128 frames, head dims 32 / 64 / 128 in
    any pair, or 16 / 16."""
    dims = (d in (32, 64, 128) and dv in (32, 64, 128)) or d == dv == 16
    return ((_MB_BWD or not bwd) and 1 <= m <= _MB_MAX_FRAMES and dims
            and all(_lstep_mb_lds(m, d, dv, last, bwd) <= _LDS_BYTES for last in (False, True)))


def _lstep_supported(m, d, dv, bwd):
    """Whether the HIP L-steps run this grid: the one-tile MFMA kernels (m <= 32, d and dv in {64, 128}), the
    multi-block MFMA kernels (m <= 128, head dims 32 / 64 / 128, or 16 / 16), or the general kernels (any m whose
    per-column tiles fit the LDS)."""
    if m <= 32 and d in (64, 128) and dv in (64, 128):
        return True
    if _lstep_mb(m, d, dv, bwd):
        return True
    return all(_lstep_general_lds(m, d, dv, last, bwd) <= _LDS_BYTES for last in (False, True))


def _fused_supported(q, k, v, num_blocks):
    D, Dv = q.shape[-1], v.shape[-1]
    # flash-entropy kernels at 64 / 128 (either dim), 32 / 32 or 16 / 16
    return (q.is_cuda and q.dtype in _lib.DTYPES and k.dtype == q.dtype and v.dtype == q.dtype
            and ((D in (64, 128) and Dv in (64, 128)) or D == Dv == 32 or D == Dv == 16)
            and _lstep_supported(num_blocks, D, Dv, False)
            and k.shape == q.shape and v.shape[:-1] == q.shape[:-1])


# Where the exact recompute of the first rt queries runs: it reads q, k, v only and writes rows [0, rt) of z, which
# the L-steps never write, so it can run beside the R/L chain.  "with_r0": its workgroups in one launch with R-step
# 0's; "start" / "after_r0" / "after_r1": on a second stream, forked there and joined at the end; "off": after the
# chain; "auto": with_r0 where that launch is built (more than one iteration, equal head dims of 64 or 128, no fp8 S)
# and 64-wide exact rows take less than _PAIR_64_MAX_FLOPS; otherwise start from _FORK_MIN_FLOPS on, else off.  Fork
# and join cost ~45 us of host time in the HIP runtime (event records and cross-stream waits), which small calls
# waited for; the shared launch costs none.  Whole
# forward, us, start / off / with_r0: 4 x 64 grid, 2 heads 59.8 / 25.7 / 21.2; 16 x 256, 8 problems 66.8 / 67.4 / 57.7;
# 21 x 400, 12 heads 150.6 / 157.1 / 151.4; 21 x 800 386.8 / 389.9 / 380.3; 33 x 993 902 / 909 / 889; 21 x 1560
# 1181 / 1194 / 1176.  At 64-wide heads R-step 0 alone has three workgroups per CU (146 registers) and in the shared
# launch two (the exact rows' 171), so there the fork wins once its host time is hidden, start / with_r0: 12 heads,
# 4 x 1200 (17.7 GFLOP of exact rows) 110 / 121, 4 x 1560 164 / 172, 33 x 700 292 / 300, 48 x 682 394 / 407, 21 x 1560
# 637 / 648, 24 heads 1265 / 1303; level at 17.2 (2 x 2048, 8 heads) 110.6 / 111.6, 33 x 400 149 / 149, 21 x 800 215 /
# 213, 21 x 1100 357 / 355; 4.0 (8 x 700, 4 heads) 64 / 55.  128-wide (two workgroups per CU either way): shared 0-9%
# faster but for 4 x 1200 (183 / 188).
_RECOMPUTE_OVERLAP = "auto"
_FORK_MIN_FLOPS = 4e9   # (~the same figures: 16 x 256, 4.3 GFLOP of exact rows, start and off are level)
_PAIR_64_MAX_FLOPS = 16e9
_OVERLAPS = {"off": 0, "start": 1, "after_r0": 2, "after_r1": 3, "with_r0": 4}
_side_streams = {}


def _side_stream(dev):
    s = _side_streams.get(dev)
    if s is None:
        s = _side_streams[dev] = torch.cuda.Stream(device=dev)   # default priority
    return s


def _vmonarch_fused(q, k, v, m, b, num_iters, recompute_tokens, min_col_mass, stage_hook=None, scale=None,
                    qk_fp8=False):
    """All-HIP forward.  `stage_hook(name, phase, stream)`, when given, is called on the host right
    before ("begin") and after ("end") each launch group ("rstep0", "lstep0", ..., "recompute") with
    the stream it goes to -- used by bench.py to bracket every kernel with events; where the recompute shares R-step
    0's launch its calls stand inside rstep0's, around the same launch.  `scale` overrides
    D ** -0.5 (q / k zero-padded past their head dim).  `qk_fp8`: the R-steps' S in fp8 (the recompute
    stays exact)."""
    B, H, N, D = q.shape
    scale = D ** -0.5 if scale is None else scale
    rt = min(int(recompute_tokens), N)
    overlap, splits = _recompute_plan(B, H, N, D, v.shape[-1], num_iters, rt, qk_fp8)
    side = _side_stream(q.device) if overlap not in (0, 4) else None
    main = torch.cuda.current_stream(q.device) if stage_hook is not None else None
    return _lib.host().vmonarch_fwd(q, k, v, m, b, num_iters, rt, min_col_mass, scale, qk_fp8, splits, overlap,
                                    side.cuda_stream if side is not None else 0, stage_hook, main, side)


def _hip_backward_supported(q, k, v, num_blocks):
    # the last R-step's backward takes the values [k | v] as two equal halves of 64 or 128
    return (_fused_supported(q, k, v, num_blocks) and q.shape[-1] == v.shape[-1]
            and _lstep_supported(num_blocks, q.shape[-1], v.shape[-1], True))


class _VMonarchFunction(torch.autograd.Function):
    """VMonarch attention with a HIP backward (the gradient autograd takes through vmonarch.py:41-69).

    The forward is the all-HIP pipeline of _vmonarch_fused, keeping what the backward needs: every
    R-step's input u, output, LSE and entropy, and the recompute's LSE.  The backward walks the
    iterations in reverse, each as the fused L-step backward (vmo_lstep_bwd) and the R-step's
    flash-entropy backward (vmo_fea_bwd on the m frames of each head, values k or [k | v]; the
    entropy enters the L-step detached, vmonarch.py:26, so its gradient is zero), then the
    recompute rows through vmo_fea_bwd (rt queries against all N keys).  Gradients of q, k, v
    collect in fp32.
    """

    @staticmethod
    def forward(ctx, q, k, v, m, b, num_iters, recompute_tokens, min_col_mass, scale=None):
        B, H, N, D = q.shape
        scale = D ** -0.5 if scale is None else scale
        rt = min(int(recompute_tokens), N)
        overlap, splits = _recompute_plan(B, H, N, D, v.shape[-1], num_iters, rt)
        ctx.orders, saved = _lib.host().vmonarch_fwd_train(
            q, k, v, m, b, num_iters, rt, min_col_mass, scale, splits, overlap,
            _side_stream(q.device).cuda_stream if overlap not in (0, 4) else 0)
        ctx.dims = (m, b, num_iters, rt, float(min_col_mass), float(scale))
        ctx.save_for_backward(*saved)
        return saved[3]

    @staticmethod
    def backward(ctx, dz):
        m, b, num_iters, rt, min_col_mass, scale = ctx.dims
        saved = ctx.saved_tensors
        D, Dv = saved[0].shape[-1], saved[2].shape[-1]
        delta = 1 if _lstep_one_tile(m, D, Dv, True) else 2 if _lstep_mb(m, D, Dv, True) else 0   # (enum Delta)
        grads = _lib.host().vmonarch_bwd(ctx.orders, saved, dz, m, b, num_iters, rt, min_col_mass, scale, delta)
        return *grads, None, None, None, None, None, None


def _vmonarch_composed(q, k, v, num_blocks, block_size, num_iters, recompute_tokens, min_col_mass):
    """Step-by-step restatement of vmonarch.py:41-69 on GPU tensors (autograd-capable)."""
    B, H, N, D = q.shape
    scale = D ** -0.5
    qg, kg, vg = (t.unflatten(2, (num_blocks, block_size)) for t in (q, k, v))
    u = qg * scale
    z = None
    for it in range(num_iters):
        last = it == num_iters - 1
        out, neg_ent = _row_block_attention(u, kg, torch.cat([kg, vg], -1) if last else kg)
        kr = out[..., :D] * scale
        logits = torch.einsum("bhijd,bhkjd->bhjik", qg, kr).float()
        attn = (logits - neg_ent.transpose(-1, -2).unsqueeze(-2)).softmax(-1)
        if last:
            y = out[..., D:]
            z = torch.einsum("bhjik,bhkjd->bhijd", attn.to(y.dtype), y)
        else:
            col_mass = attn.sum(-2).transpose(-1, -2).clamp_min(min_col_mass)
            u = torch.einsum("bhjik,bhijd->bhkjd", attn.to(q.dtype), qg)
            u = u * (scale / col_mass.unsqueeze(-1)).to(q.dtype)
    z = z.reshape(B, H, N, -1)
    if recompute_tokens > 0:
        exact = torch.nn.functional.scaled_dot_product_attention(q[:, :, :recompute_tokens], k, v)
        z = torch.cat([exact, z[:, :, recompute_tokens:]], dim=2)
    return z


def _padded_width(D, Dv):
    """The kernel width (32, 64 or 128) that q, k and v can all be zero-padded to, or None."""
    if D <= 32 and Dv <= 32:
        return 32
    w = max(64, D, Dv)
    return w if w in (64, 128) else None


def _pad_to(t, w):
    return t if t.shape[-1] == w else torch.nn.functional.pad(t, (0, w - t.shape[-1]))


def vmonarch_attention(q, k, v, num_blocks, block_size, num_iters=2, recompute_tokens=0, min_col_mass=0.01,
                       qk_fp8=False):
    """
    Args:
        q, k: (B, H, N, D); v: (B, H, N, Dv), with N == num_blocks * block_size.
        num_blocks: m, number of grid rows (keep it small).
        block_size: b, number of tokens per grid row.
        num_iters: alternating-minimization steps.
        recompute_tokens: the first `recompute_tokens` queries use exact attention.
        min_col_mass: lower bound of the column mass of L, for stability.
        qk_fp8: (beyond the reference) the R-steps' q k^T in fp8 e4m3, forward only, D = 128; the
            recompute stays exact.  An approximation: logits off by ~1% of their spread.  D = Dv = 128.
    Returns:
        (B, H, N, Dv)
    """
    B, H, N, D = q.shape
    assert N == num_blocks * block_size, f"N={N} != {num_blocks} * {block_size}"
    if num_iters < 1:
        raise UnboundLocalError("local variable 'z' referenced before assignment")  # as the reference (vmonarch.py:65)
    needs_graph = torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v))
    Dv = v.shape[-1]
    if qk_fp8:
        if needs_graph:
            raise NotImplementedError("vmonarch_amd: qk_fp8 is forward-only (the backward recomputes S in the "
                                      "16-bit type); run under torch.no_grad() or without it")
        if not (_row_block_attention is _ROW_BLOCK_ATTENTION and D == 128 and Dv == 128
                and _fused_supported(q, k, v, num_blocks)):
            raise NotImplementedError(f"vmonarch_amd: qk_fp8 is built for the fused HIP path with head dim 128 "
                                      f"(got D={D}, Dv={Dv}, num_blocks={num_blocks}, {q.dtype})")
        return _vmonarch_fused(q, k, v, num_blocks, block_size, num_iters, recompute_tokens, min_col_mass,
                               qk_fp8=True)
    if _row_block_attention is _ROW_BLOCK_ATTENTION:
        args = (num_blocks, block_size, num_iters, recompute_tokens, min_col_mass)
        if not needs_graph and _fused_supported(q, k, v, num_blocks):
            return _vmonarch_fused(q, k, v, *args)
        if needs_graph and _hip_backward_supported(q, k, v, num_blocks):
            return _VMonarchFunction.apply(q, k, v, *args)
        # Head dims the kernels do not take as they are (mixes of 16 and 32, or D != Dv with autograd): zero columns
        # change neither q.k nor P.v, so q, k and v padded to one kernel width give z with zero columns
        # past Dv, with the softmax scale of the true D; autograd slices the padded gradients back.
        w = _padded_width(D, Dv)
        if (w is not None and q.is_cuda and q.dtype in _lib.DTYPES and k.dtype == q.dtype and v.dtype == q.dtype
                and k.shape == q.shape and v.shape[:-1] == q.shape[:-1]
                and _lstep_supported(num_blocks, w, w, needs_graph)):
            qp, kp, vp = (_pad_to(t, w) for t in (q, k, v))
            if needs_graph:
                z = _VMonarchFunction.apply(qp, kp, vp, *args, D ** -0.5)
            else:
                z = _vmonarch_fused(qp, kp, vp, *args, scale=D ** -0.5)
            if w == Dv:
                return z
            # the first Dv columns, in the caller's memory order like every other path's z (a DiT block's
            # (B, N, H, Dv) buffer needs no permute copy afterwards); copy_ keeps the autograd graph
            return _lib.empty_in_layout(q, Dv, q.dtype).copy_(z[..., :Dv])
        if q.is_cuda:
            warnings.warn(f"vmonarch_amd: no HIP path for num_blocks={num_blocks}, head dims ({D}, {Dv}), {q.dtype}"
                          f"{' with autograd' if needs_graph else ''}; running the composed path (flash-entropy "
                          "R-steps in HIP, L-steps and recompute as torch ops)", RuntimeWarning, stacklevel=2)
    if not q.is_cuda:
        raise RuntimeError("vmonarch_amd: vmonarch_attention needs GPU tensors (no CPU path)")
    return _vmonarch_composed(q, k, v, num_blocks, block_size, num_iters, recompute_tokens, min_col_mass)


class VMonarchAttention(nn.Module):
    """Module wrapper (reference vmonarch.py:72-85); holds no parameters."""

    def __init__(self, num_blocks, block_size, num_iters=2, min_col_mass=0.01, qk_fp8=False):
        super().__init__()
        self.num_blocks = num_blocks
        self.block_size = block_size
        self.num_iters = num_iters
        self.min_col_mass = min_col_mass
        self.qk_fp8 = qk_fp8   # beyond the reference: fp8 q k^T in the R-steps (vmonarch_attention)

    def forward(self, q, k, v, recompute_tokens=0):
        return vmonarch_attention(q, k, v, self.num_blocks, self.block_size, self.num_iters,
                                  recompute_tokens, self.min_col_mass, qk_fp8=self.qk_fp8)

    def extra_repr(self):
        return f"num_blocks={self.num_blocks}, block_size={self.block_size}, num_iters={self.num_iters}"
