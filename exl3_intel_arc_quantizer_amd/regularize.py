"""Weight regularisation before LDLQ, as a three-pass GPU pipeline
(reference: exl3_quant/regularize.py:41-211; public names and signatures kept).

What the transform is (fixed by the EXL3 format, because decoding undoes it
in reverse with ``hadamard.weight_from_quantized``): a (k, n) weight W
becomes ``H_l((H_r(W / sv)) / su) * g``, where

* sv (1, n) carries the output-channel scales: the RMS of each column of W
  divided by the mean column RMS, plus 1e-10, when the Hessian diagonal is
  not too skewed (the top 2 % of sqrt(diag H) hold less than 15 % of its
  sum), else the caller's sv unchanged; columns whose RMS is zero keep a
  0.1 scale for the division and are stored as sv = 0;
* su (k, 1) carries the input-channel scales: the RMS of each row of
  H_r(W / sv), divided by -1.24371088 (the codebook's scale), plus 1e-10;
  zero rows use 0.1;
* g is the global scale (1 unless a search function is given).

How it runs here. The reference spends about a dozen full passes over the
matrix (clone, RMS, division, transform, RMS, division, transform). This
module makes three, on HIP kernels of ``libexl3_hip.so``:

1. ``exl3_output_scales``: the column RMS of W, its mean, the skew of the
   Hessian diagonal (radix selection of its largest 2 %) and sv, every
   decision taken on the device;
2. ``exl3_row_energy``: the sums of squares of the rows of W / sv, which the
   right transform keeps, in 128-element segments; ``exl3_input_scales``
   turns those into the row RMS and su;
3. ``exl3_rotate``: both divisions and both transforms of a 128 x 128 block in
   one read and one write.

The decisions (any energy, skew, scales applied) come back in one read after
the last pass. A 4096 x 4096 weight takes 119 us, where torch operations on
the scale vectors between the passes, a sort of the diagonal and strided
reductions took 322 us.

Rounding. Divisions are correctly rounded fp32, like torch's; the transform
is the fast Walsh-Hadamard transform of ``exl3_hadamard128``. The column RMS
sums 32-row slices in order and adds them in slice order, as the reference's
``block_rms`` does; the row RMS adds the sums of 128-element segments in order,
each a butterfly over lanes, and takes them before the orthonormal transform
instead of after it, which leaves out the transform's roundings.
Results therefore agree with the reference's to float32 rounding.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Callable, Optional, Tuple

import torch

from .hadamard import HAD_DIM, records

# The values of the kernels of exl3_output_scales / exl3_input_scales.
CODEBOOK_SCALE = 1.24371088     # the codebook's RMS, regularize.py:33
OUT_SCALE_SKEW_CUTOFF = 0.15    # output scales only below this skew
SKEW_FRACTION = 50              # the skew looks at the top 1/50 of the diagonal
ZERO_FLOOR = 0.1                # scale used for an all-zero row or column
EPS = 1e-10                     # added to every scale
RMS_SLICE = 32                  # block_rms slice length


def block_rms(x: torch.Tensor, dim: int, keepdim: bool = False,
              blocksize: int = RMS_SLICE) -> torch.Tensor:
    """Root mean square along ``dim`` of a 2-D GPU tensor (regularize.py:41-56):
    squares summed in ``blocksize`` slices, slice sums added in slice order,
    one launch pair of ``exl3_block_rms``."""
    if x.dim() != 2:
        raise ValueError(f"block_rms expects a 2-D tensor, got shape {tuple(x.shape)}")
    if x.device.type != "cuda":
        raise ValueError("block_rms runs on the GPU; move the tensor to a cuda device")
    from ._native import block_rms as _block_rms
    axis = dim % 2
    rows, cols = x.shape
    src = x if (x.dtype == torch.float32 and x.is_contiguous()) else \
        x.to(torch.float32).contiguous()
    n_out = cols if axis == 0 else rows
    out = torch.empty(n_out, dtype=torch.float32, device=x.device)
    _block_rms(src, out, axis, int(blocksize))
    if keepdim:
        return out.reshape(1, cols) if axis == 0 else out.reshape(rows, 1)
    return out


@dataclass
class RegularizeResult:
    """Outputs of :func:`regularize` (regularize.py:59-71)."""

    apply_out_scales: bool
    weight: torch.Tensor
    g_scale: float
    su: torch.Tensor
    sv: torch.Tensor
    out_channel_scales: torch.Tensor
    in_channel_scales: torch.Tensor
    zeros: bool
    skew_factor: Optional[float]


def _skew_tensor(H_diag: torch.Tensor) -> torch.Tensor:
    root = torch.sort(H_diag.sqrt(), descending=True).values
    top = root.shape[0] // SKEW_FRACTION
    return root[:top].sum() / root.sum()


def hessian_skew(H_diag: torch.Tensor) -> float:
    """Share of sum(sqrt(diag H)) held by its largest len/50 entries."""
    return float(_skew_tensor(H_diag))


def _out_scale_decision(H_diag: Optional[torch.Tensor], forced: Optional[bool],
                        q_fallback: bool) -> Tuple[Optional[bool], bool]:
    """(apply the output-channel scales?, is the skew wanted?). A forced
    value wins; without one the skew decides, and without a Hessian diagonal
    the scales apply. In fallback mode only a forced True applies them. The
    decision is None when the skew makes it: it is then taken on the device
    and read back once, at the end."""
    if q_fallback:
        return bool(forced), False
    if H_diag is None:
        return (True if forced is None else bool(forced)), False
    return (None if forced is None else bool(forced)), True


def _check_inputs(weight: torch.Tensor, su: torch.Tensor, sv: torch.Tensor, had_dim: int) -> None:
    if weight.dim() != 2:
        raise ValueError(f"weight must be 2-D, got shape {tuple(weight.shape)}")
    if weight.dtype != torch.float32:
        raise ValueError(f"weight must be float32, got {weight.dtype}")
    k, n = weight.shape
    if su.numel() != k or sv.numel() != n:
        raise ValueError(f"su must have {k} elements and sv {n}, got {su.numel()} / {sv.numel()}")
    if k % had_dim != 0 or n % had_dim != 0:
        raise ValueError(f"both dimensions must be divisible by {had_dim}, got {(k, n)}")
    if had_dim != HAD_DIM:
        raise ValueError(f"only had_dim={HAD_DIM} is supported, got {had_dim}")
    if weight.device.type != "cuda":
        raise ValueError("regularize runs on the GPU; move the weight to a cuda device")


def regularize(weight: torch.Tensor, su: torch.Tensor, sv: torch.Tensor,
               quant_args: Optional[dict] = None, H_diag: Optional[torch.Tensor] = None,
               skip_g_scale: bool = True, q_fallback: bool = False,
               g_scale_fn: Optional[Callable[[torch.Tensor], float]] = None,
               had_dim: int = HAD_DIM) -> RegularizeResult:
    """Transform a (k, n) float32 GPU weight into the encoder's basis
    (regularize.py:83-211). ``weight`` is not modified. ``quant_args`` may
    force ``apply_out_scales``; when given, its ``zeros`` entry is set to
    whether W had no energy at all."""
    from ._native import input_scales, output_scales, rotate, row_energy

    _check_inputs(weight, su, sv, had_dim)
    k, n = weight.shape
    dev = weight.device
    forced = None if quant_args is None else quant_args.get("apply_out_scales")
    apply_out, skew_needed = _out_scale_decision(H_diag, forced, q_fallback)
    w = weight.contiguous()

    # Pass 1: output-channel scales from the column RMS, normalised by their
    # mean unless W has no energy (the scales then stay as they are). Nothing
    # is read back here: the decisions are taken on the device and come back
    # together after the last pass.
    vec = dict(dtype=torch.float32, device=dev)
    out_scales = torch.empty((1, n), **vec)
    divisor, sv_out = torch.empty(n, **vec), torch.empty((1, n), **vec)
    flags = torch.zeros(3, dtype=torch.float64, device=dev)
    sv = sv.to(device=dev, dtype=torch.float32).reshape(n).contiguous()
    diag = None
    if skew_needed:
        if H_diag.dtype == torch.float32 and H_diag.device == dev and H_diag.dim() == 1 \
                and H_diag.numel() > 0 and H_diag.stride(0) > 0:
            diag = H_diag
        else:
            flags[1] = _skew_tensor(H_diag)
    # Where torch follows sv, the kernel works on ones and sv is folded by
    # torch's operations, to the same values.
    follow_sv = records(sv)
    output_scales(w, torch.ones_like(sv) if follow_sv else sv,
                  2 if apply_out is None else int(apply_out), forced is not None,
                  out_scales, divisor, sv_out, flags, diag)
    if follow_sv:
        dead_cols = sv_out == 0.0
        sv = sv.reshape(1, n)
        sv_out = torch.where(flags[2] != 0.0, (sv * out_scales + EPS).float(), sv)
        divisor = sv_out.detach().reshape(n).clone()
        sv_out = sv_out.masked_fill(dead_cols, 0.0)

    # Pass 2: the row sums of squares of W / sv (and so of its right
    # transform, which is orthonormal) for the input-channel scales.
    energy = torch.empty((k, n // HAD_DIM), **vec)
    row_energy(w, divisor, energy)
    in_scales, su_out = torch.empty((k, 1), **vec), torch.empty((k, 1), **vec)
    su = su.to(device=dev, dtype=torch.float32).reshape(k).contiguous()
    input_scales(energy, su, in_scales, su_out, n)
    if records(su):
        su_out = (su.reshape(k, 1) * in_scales / (-CODEBOOK_SCALE) + EPS).float()

    # Pass 3: both divisions and both transforms.
    work = torch.empty_like(w)
    rotate(w, divisor, su_out, work)

    if skip_g_scale:
        g_scale = 1.0
    else:
        if g_scale_fn is None:
            raise ValueError("skip_g_scale=False requires g_scale_fn")
        g_scale = float(g_scale_fn(work))
        if not g_scale > 0.0:
            raise ValueError(f"g_scale_fn returned a non-positive scale: {g_scale}")
        work *= g_scale
        su_out /= g_scale
    live, skew, applied = flags.tolist()         # the one read-back of the pipeline
    zeros = not live
    if quant_args is not None:
        quant_args["zeros"] = zeros
    return RegularizeResult(apply_out_scales=bool(applied), weight=work, g_scale=g_scale,
                            su=su_out, sv=sv_out, out_channel_scales=out_scales,
                            in_channel_scales=in_scales, zeros=zeros,
                            skew_factor=skew if skew_needed else None)

