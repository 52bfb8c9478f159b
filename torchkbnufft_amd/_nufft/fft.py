"""Oversampled FFT stages: the fused HIP FFT, or fused scale/pad and crop/deapodise around torch.fft.

``fft_and_scale`` / ``ifft_and_scale`` keep the signatures of
``torchkbnufft/_nufft/fft.py:36-118``.  The element-wise work (scaling, zero-pad,
crop, conjugate scaling, the SENSE coil expansion and coil combine of
``modules/kbnufft.py:182-183,404-405``) is part of the FFT's first and last pass
(complex64, any grid size within the limits of ``tkbn_fft_any_supported``), or one HIP
pass on each side of an unnormalised ``torch.fft`` (complex128, larger sizes); the
``"ortho"`` factor is folded in.
"""
from __future__ import annotations

import ctypes
import math
from typing import Optional

import torch
from torch import Tensor

from .. import _lib
from .._autograd._apply import run as _run
from ._host import host_values, plain, plain_as, require_gpu


def _norm_scale(norm: Optional[str], grid_size) -> float:
    if norm is None:
        return 1.0
    if norm == "ortho":
        return 1.0 / math.sqrt(float(math.prod(int(v) for v in grid_size)))
    raise ValueError("Only option for norm is 'ortho'.")


def apod_pad(image: Tensor, smaps: Optional[Tensor], scaling_coef: Tensor, im_size, grid_size, scale: float) -> Tensor:
    """grid[b, c] = pad_end(image[b, c or 0] * smaps[b, c] * scaling_coef) * scale."""
    require_gpu(image, smaps, scaling_coef)
    image = plain(image)
    im = tuple(int(v) for v in im_size)
    gs = tuple(int(v) for v in grid_size)
    d = len(im)
    B = image.shape[0]
    C = smaps.shape[1] if smaps is not None else image.shape[1]
    if tuple(image.shape[2:]) != im:
        raise ValueError(f"image spatial shape {tuple(image.shape[2:])} != im_size {im}")
    if smaps is not None:
        smaps = plain(smaps.to(image.dtype))
        if tuple(smaps.shape) != (B, C) + im and not (smaps.shape[0] == 1 and tuple(smaps.shape[1:]) == (C,) + im):
            raise ValueError(f"smaps shape {tuple(smaps.shape)} does not match image {tuple(image.shape)}")
        if smaps.shape[0] != B:
            smaps = smaps.expand(B, *smaps.shape[1:]).contiguous()
        if image.shape[1] not in (1, C):
            raise ValueError("image coil dimension must be 1 or match smaps")
    sc = plain_as(scaling_coef, image, image.dtype)
    if sc.numel() != math.prod(im):
        raise ValueError("scaling_coef does not match im_size")
    grid = torch.empty((B, C) + gs, dtype=image.dtype, device=image.device)
    with _lib.on_device(image):
        st = _lib.load().tkbn_apod_pad(
            _lib.dtype_code(image),
            d,
            _lib.i64_array(im),
            _lib.i64_array(gs),
            B,
            C,
            image.shape[1],
            image.data_ptr(),
            smaps.data_ptr() if smaps is not None else None,
            sc.data_ptr(),
            float(scale),
            grid.data_ptr(),
            _lib.stream_of(image),
        )
    _lib.check(st, "tkbn_apod_pad")
    return grid


def crop_deapod(grid: Tensor, smaps: Optional[Tensor], scaling_coef: Tensor, im_size, scale: float) -> Tensor:
    """image[b, c] = crop(grid[b, c]) * conj(scaling_coef) * scale; with smaps summed
    over coils against conj(smaps) into image[b, 0]."""
    require_gpu(grid, smaps, scaling_coef)
    grid = plain(grid)
    im = tuple(int(v) for v in im_size)
    d = len(im)
    gs = tuple(grid.shape[2:])
    B, C = grid.shape[0], grid.shape[1]
    if smaps is not None:
        smaps = plain(smaps.to(grid.dtype))
        if smaps.shape[0] != B:
            smaps = smaps.expand(B, *smaps.shape[1:]).contiguous()
        if tuple(smaps.shape) != (B, C) + im:
            raise ValueError(f"smaps shape {tuple(smaps.shape)} does not match data ({B}, {C}) + {im}")
    sc = plain_as(scaling_coef, grid, grid.dtype)
    out = torch.empty((B, 1 if smaps is not None else C) + im, dtype=grid.dtype, device=grid.device)
    _crop_deapod_into(grid, smaps, sc, im, scale, out)
    return out


def _crop_deapod_into(grid: Tensor, smaps: Optional[Tensor], sc: Tensor, im, scale: float, out: Tensor) -> None:
    d, gs = len(im), tuple(grid.shape[2:])
    B, C = grid.shape[0], grid.shape[1]
    with _lib.on_device(grid):
        st = _lib.load().tkbn_crop_deapod(
            _lib.dtype_code(grid),
            d,
            _lib.i64_array(im),
            _lib.i64_array(gs),
            B,
            C,
            grid.data_ptr(),
            smaps.data_ptr() if smaps is not None else None,
            sc.data_ptr(),
            float(scale),
            out.data_ptr(),
            _lib.stream_of(grid),
        )
    _lib.check(st, "tkbn_crop_deapod")


def fft_and_scale(image: Tensor, scaling_coef: Tensor, im_size: Tensor, grid_size: Tensor, norm: Optional[str] = None) -> Tensor:
    """Oversampled FFT of ``image * scaling_coef`` (``fft.py:36-76``)."""
    from .._autograd.fft import ApodPad, GridForward

    gs = host_values(grid_size)
    im = host_values(im_size)
    scale = _norm_scale(norm, gs)
    if pipeline_supported(image.dtype, im, gs):
        return _run(GridForward, image, None, scaling_coef, im, gs, scale)
    grid = _run(ApodPad, image, None, scaling_coef, im, gs, scale)
    return torch.fft.fftn(grid, dim=tuple(range(-len(gs), 0)), norm="backward")


def ifft_and_scale(image: Tensor, scaling_coef: Tensor, im_size: Tensor, grid_size: Tensor, norm: Optional[str] = None) -> Tensor:
    """Unnormalised (or ortho) inverse FFT, crop, conjugate scaling (``fft.py:80-118``)."""
    from .._autograd.fft import CropDeapod, GridAdjoint

    gs = host_values(grid_size)
    im = host_values(im_size)
    scale = _norm_scale(norm, gs)
    if pipeline_supported(image.dtype, im, gs):
        return _run(GridAdjoint, image, None, scaling_coef, im, scale)
    x = torch.fft.ifftn(image, dim=tuple(range(-len(gs), 0)), norm="forward")
    return _run(CropDeapod, x, None, scaling_coef, im, scale)


# ---------------------------------------------------------------------------
# fused FFT path (complex64, grid sizes with prime factors 2, 3, 5)
# ---------------------------------------------------------------------------
_FUSED_OK = {}
_FUSED_DISABLED = False


def set_fused_fft(enabled: bool) -> None:
    """Use the fused HIP FFT where the geometry allows (default) or always torch.fft."""
    global _FUSED_DISABLED
    _FUSED_DISABLED = not enabled


def fused_supported(dtype: torch.dtype, im_size, grid_size) -> bool:
    if _FUSED_DISABLED or dtype != torch.complex64:
        return False
    key = (tuple(int(v) for v in im_size), tuple(int(v) for v in grid_size))
    ok = _FUSED_OK.get(key)
    if ok is None:
        d = len(key[0])
        ok = _lib.load().tkbn_fft_supported(d, _lib.i64_array(key[0]), _lib.i64_array(key[1])) == _lib.TKBN_OK
        _FUSED_OK[key] = ok
    return ok


def pipeline_supported(dtype: torch.dtype, im_size, grid_size) -> bool:
    """The fused FFT, or the same passes with the other grid sizes as convolutions."""
    if fused_supported(dtype, im_size, grid_size):
        return True
    if _FUSED_DISABLED or dtype != torch.complex64:
        return False
    key = (tuple(int(v) for v in im_size), tuple(int(v) for v in grid_size), "any")
    ok = _FUSED_OK.get(key)
    if ok is None:
        ok = (
            _lib.load().tkbn_fft_any_supported(len(key[0]), _lib.i64_array(key[0]), _lib.i64_array(key[1]))
            == _lib.TKBN_OK
        )
        _FUSED_OK[key] = ok
    return ok


def _smooth(im, gs) -> bool:
    """Every extent has compiled or planned butterflies (whatever set_fused_fft says)."""
    key = (tuple(im), tuple(gs))
    ok = _FUSED_OK.get(key)
    if ok is None:
        ok = _lib.load().tkbn_fft_supported(len(key[0]), _lib.i64_array(key[0]), _lib.i64_array(key[1])) == _lib.TKBN_OK
        _FUSED_OK[key] = ok
    return ok


def _combines(im, gs, B: int, C: int) -> bool:
    """The adjoint's last pass sums the coils itself on a grid of any factors: where the last
    dimension is no convolution (a line's workspace then holds no chirp, as that of one value),
    and where a group per line of the image, which takes the coils in turn, is no slower than
    the coils' images apart and summed by another kernel.  That is up to 800 values a line
    (longer ones leave a group few coils at once: 8 coils, 490^2 -> 980^2 88 us apart, 94 combined,
    385^2 -> 770^2 65 and 52), with a group for every CU or no more than one round of coils
    (32 coils, 182^2 -> 364^2 42 and 48; 12 coils 28 and 24; 308^2 -> 616^2 119 and 85)."""
    if int(gs[-1]) > 800 or (C > 16 and B * math.prod(int(n) for n in im[:-1]) < 256):
        return False
    key = (int(im[-1]), int(gs[-1]), "combine")
    ok = _FUSED_OK.get(key)
    if ok is None:
        size = _lib.load().tkbn_fft_any_workspace_bytes
        ok = size(1, _lib.i64_array(key[:1]), _lib.i64_array(key[1:2]), 1, 1) == size(1, _lib.i64_array([1]), _lib.i64_array([1]), 1, 1)
        _FUSED_OK[key] = ok
    return ok


def _out_or_new(out: Optional[Tensor], shape: tuple, like: Tensor) -> Tensor:
    if out is None:
        return torch.empty(shape, dtype=like.dtype, device=like.device)
    if tuple(out.shape) != tuple(shape) or out.dtype != like.dtype or out.device != like.device or not out.is_contiguous():
        raise ValueError(f"out must be a contiguous {tuple(shape)} {like.dtype} tensor on {like.device}")
    return out


def _fft_workspace(dev, d, im, gs, B, C, smooth=True):
    lib = _lib.load()
    n = (lib.tkbn_fft_workspace_bytes if smooth else lib.tkbn_fft_any_workspace_bytes)(d, _lib.i64_array(im), _lib.i64_array(gs), B, C)
    if n < 0:
        _lib.check(_lib.TKBN_ERR_INVALID, "tkbn_fft_workspace_bytes")
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device=dev), int(n)


def fft_grid_fwd(image: Tensor, smaps: Optional[Tensor], scaling_coef: Tensor, im_size, grid_size, scale: float,
                 out: Optional[Tensor] = None) -> Tensor:
    """FFT(pad_end(image * smaps * scaling_coef)) * scale in one fused HIP pipeline."""
    require_gpu(image, smaps, scaling_coef)
    image = plain(image)
    im = tuple(int(v) for v in im_size)
    gs = tuple(int(v) for v in grid_size)
    d = len(im)
    B = image.shape[0]
    C = smaps.shape[1] if smaps is not None else image.shape[1]
    if tuple(image.shape[2:]) != im:
        raise ValueError(f"image spatial shape {tuple(image.shape[2:])} != im_size {im}")
    if smaps is not None:
        smaps = smaps.to(image.dtype)
        if smaps.shape[0] != B:
            smaps = smaps.expand(B, *smaps.shape[1:])
        smaps = plain(smaps)
        if tuple(smaps.shape) != (B, C) + im:
            raise ValueError(f"smaps shape {tuple(smaps.shape)} does not match image {tuple(image.shape)}")
        if image.shape[1] not in (1, C):
            raise ValueError("image coil dimension must be 1 or match smaps")
    sc = plain_as(scaling_coef, image, image.dtype)
    grid = _out_or_new(out, (B, C) + gs, image)
    smooth = _smooth(im, gs)
    ws, nws = _fft_workspace(image.device, d, im, gs, B, C, smooth)
    lib = _lib.load()
    with _lib.on_device(image):
        st = (lib.tkbn_fft_grid_fwd if smooth else lib.tkbn_fft_any_grid_fwd)(
            _lib.dtype_code(image), d, _lib.i64_array(im), _lib.i64_array(gs), B, C, image.shape[1],
            image.data_ptr(), smaps.data_ptr() if smaps is not None else None, sc.data_ptr(), float(scale),
            grid.data_ptr(), ws.data_ptr(), nws, _lib.stream_of(image),
        )
    _lib.check(st, "tkbn_fft_grid_fwd")
    return grid


def fft_grid_adj(grid: Tensor, smaps: Optional[Tensor], scaling_coef: Tensor, im_size, scale: float,
                 out: Optional[Tensor] = None) -> Tensor:
    """sum_c crop(IFFT(grid)) * conj(scaling_coef) * conj(smaps_c) * scale (per coil without smaps)."""
    require_gpu(grid, smaps, scaling_coef)
    grid = plain(grid)
    im = tuple(int(v) for v in im_size)
    gs = tuple(grid.shape[2:])
    d = len(im)
    B, C = grid.shape[0], grid.shape[1]
    if smaps is not None:
        smaps = smaps.to(grid.dtype)
        if smaps.shape[0] != B:
            smaps = smaps.expand(B, *smaps.shape[1:])
        smaps = plain(smaps)
        if tuple(smaps.shape) != (B, C) + im:
            raise ValueError(f"smaps shape {tuple(smaps.shape)} does not match data ({B}, {C}) + {im}")
    sc = plain_as(scaling_coef, grid, grid.dtype)
    smooth = _smooth(im, gs)
    combine = smaps is not None and not smooth and not _combines(im, gs, B, C)
    out = _out_or_new(out, (B, 1 if smaps is not None else C) + im, grid)
    image = torch.empty((B, C) + im, dtype=grid.dtype, device=grid.device) if combine else out
    ws, nws = _fft_workspace(grid.device, d, im, gs, B, C, smooth)
    lib = _lib.load()
    with _lib.on_device(grid):
        st = (lib.tkbn_fft_grid_adj if smooth else lib.tkbn_fft_any_grid_adj)(
            _lib.dtype_code(grid), d, _lib.i64_array(im), _lib.i64_array(gs), B, C, grid.data_ptr(),
            smaps.data_ptr() if smaps is not None and not combine else None, None if combine else sc.data_ptr(),
            1.0 if combine else float(scale), image.data_ptr(), ws.data_ptr(), nws, _lib.stream_of(grid),
        )
    _lib.check(st, "tkbn_fft_grid_adj")
    if combine:
        _crop_deapod_into(image, smaps, sc, im, scale, out)
    return out


# ---------------------------------------------------------------------------
# FFT filtering on an oversampled grid (Toeplitz embedding)
# ---------------------------------------------------------------------------
_ONES = {}


def _ones_scaling(im, dtype, device) -> Tensor:
    key = (tuple(im), dtype, device)
    t = _ONES.get(key)
    if t is None:
        t = torch.ones(tuple(im), dtype=dtype, device=device)
        _ONES[key] = t
    return t


def fft_filter_fused(image: Tensor, smaps: Optional[Tensor], kernel: Tensor, kernel_batched: bool,
                     scale_fwd: float, scale_adj: float) -> Tensor:
    """One tkbn_fft_filter call: image (B, 1|C, *N) [, smaps (B|1, C, *N)], kernel
    (*K) or (B, *K) with kernel_batched; returns (B, 1|C, *N)."""
    require_gpu(image, smaps, kernel)
    image = plain(image)
    d = image.ndim - 2
    im = tuple(int(v) for v in image.shape[2:])
    gs = tuple(int(v) for v in kernel.shape[-d:])
    B = image.shape[0]
    C = smaps.shape[1] if smaps is not None else image.shape[1]
    if smaps is not None:
        smaps = smaps.to(image.dtype)
        if smaps.shape[0] != B:
            smaps = smaps.expand(B, *smaps.shape[1:])
        smaps = plain(smaps)
        if tuple(smaps.shape) != (B, C) + im:
            raise ValueError(f"smaps shape {tuple(smaps.shape)} does not match image {tuple(image.shape)}")
    kernel = plain(kernel.to(image.dtype))
    if kernel.numel() != (B if kernel_batched else 1) * math.prod(gs):
        raise ValueError(f"kernel of shape {tuple(kernel.shape)} does not match batch {B} and grid {gs}")
    out = torch.empty((B, 1 if smaps is not None else C) + im, dtype=image.dtype, device=image.device)
    ws, nws = _fft_workspace(image.device, d, im, gs, B, C)
    with _lib.on_device(image):
        st = _lib.load().tkbn_fft_filter(
            _lib.dtype_code(image), d, _lib.i64_array(im), _lib.i64_array(gs), B, C, image.shape[1],
            image.data_ptr(), smaps.data_ptr() if smaps is not None else None, kernel.data_ptr(),
            1 if kernel_batched else 0, float(scale_fwd), float(scale_adj), out.data_ptr(), ws.data_ptr(), nws,
            _lib.stream_of(image),
        )
    _lib.check(st, "tkbn_fft_filter")
    return out


def toeplitz_filter(image: Tensor, smaps: Optional[Tensor], kernel: Tensor, norm: Optional[str]) -> Tensor:
    """crop(iFFT(kernel * FFT(pad_end(image [* smaps])))) [summed against conj(smaps)].

    The grid size is the kernel's trailing extents.  Where the fused FFT covers the
    geometry (complex64, 2/3/5-smooth sizes, two or more dimensions) the whole
    operator is one tkbn_fft_filter pipeline: the padded grid is never written
    (dimension 0 is transformed, multiplied by the kernel and transformed back in one
    pass).  One-dimensional problems, or a kernel or smaps that needs a gradient, use
    the fused pad + FFT and iFFT + crop stages with the product in between; other
    geometries use rocFFT.
    """
    from .._autograd.fft import FftFilter, GridAdjoint, GridForward

    if norm is not None and norm != "ortho":
        raise ValueError("Only option for norm is 'ortho'.")
    require_gpu(image, smaps, kernel)
    d = image.ndim - 2
    im = tuple(int(v) for v in image.shape[2:])
    gs = tuple(int(v) for v in kernel.shape[-d:])
    scale = _norm_scale(norm, gs)
    fused = fused_supported(image.dtype, im, gs) and all(g >= n for g, n in zip(gs, im))
    lead = tuple(kernel.shape[:-d])
    one_pass = (
        fused
        and d >= 2
        and kernel.dtype == image.dtype
        and (lead == () or (smaps is not None and lead == (image.shape[0], 1)))
        and not (torch.is_grad_enabled() and (kernel.requires_grad or (smaps is not None and smaps.requires_grad)))
    )
    if one_pass:
        return _run(FftFilter, image, smaps, kernel, lead != (), scale, scale)
    if fused:
        ones = _ones_scaling(im, image.dtype, image.device)
        grid = _run(GridForward, image, smaps, ones, im, gs, scale)
        return _run(GridAdjoint, grid * kernel, smaps, ones, im, scale)
    x = image * smaps if smaps is not None else image
    pad = []
    for g, n in zip(reversed(gs), reversed(im)):
        pad += [0, g - n]
    dims = tuple(range(-d, 0))
    grid = torch.fft.fftn(torch.nn.functional.pad(x, pad), dim=dims, norm="ortho" if norm == "ortho" else None)
    x = torch.fft.ifftn(grid * kernel, dim=dims, norm="ortho" if norm == "ortho" else "forward")
    for ax, n in enumerate(im):
        x = x.narrow(2 + ax, 0, n)
    if smaps is not None:
        x = torch.sum(x * smaps.conj(), dim=1, keepdim=True)
    return x


def fft_filter(image: Tensor, kernel: Tensor, norm: Optional[str] = "ortho") -> Tensor:
    """``iFFT(kernel * FFT(image))`` on an oversampled grid (``fft.py:121-173``)."""
    return toeplitz_filter(image, None, kernel, norm)
