"""Token merge / split operators on HIP kernels.

Same names, argument meaning and return values as the reference's pybind module
``co_me_cuext`` (``src/cuda_extension/co_me/src/binding.cpp:33-51``,
``co_me_cuext.pyi:8-58``); argument errors raise ``RuntimeError`` as ``TORCH_CHECK``
does there (``kernel_token_merge.cu:246-261, 360-363``).  Unlike the reference the
kernels run on the current HIP stream of the tensors' device.

Two additional operators have no counterpart in the reference: the 2-D window
merge without a permuted copy (``co_me_token_merge_2d_cuda``) and the fused
confidence selection + merge (``co_me_select_merge_2d``).
"""

from __future__ import annotations

import torch

from ... import _lib

__all__ = [
    "co_me_token_merge_cuda",
    "co_me_token_split_cuda",
    "co_me_token_split_pair_cuda",
    "co_me_token_merge_2d_cuda",
    "co_me_select_windows",
    "co_me_select_merge_2d",
]


def _torch_check(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


def co_me_token_merge_cuda(tokens: torch.Tensor, start_index: int, group_size: int, merge_mask: torch.Tensor):
    """Fused token merge: ``(tokens [B,N,C], start_index, G, merge_mask [B,M] bool)`` ->
    ``(out_flat [P,C], offsets [B+1] int32, rev_id [B*N] int64, weight [P] float32)``."""
    _torch_check(tokens.is_cuda, "tokens must be on CUDA")
    _torch_check(merge_mask.is_cuda, "merge_mask must be on CUDA")
    _torch_check(tokens.dim() == 3, "tokens must be [B, N, C]")
    _torch_check(merge_mask.dim() == 2, "merge_mask must be [B, M]")
    start_index, group_size = int(start_index), int(group_size)
    mask = merge_mask if merge_mask.dtype == torch.bool else merge_mask.to(torch.bool)
    merged = _lib.host().merge_1d(tokens, start_index, group_size, mask, False)
    if merged is None:
        B, N, _ = tokens.shape
        _torch_check(mask.shape[0] == B, "merge_mask batch != tokens batch")
        _torch_check(start_index >= 0 and group_size > 0, "start_index must be >= 0 and group_size > 0")
        _torch_check(N == start_index + mask.shape[1] * group_size, "N != start_index + M * group_size")
        _torch_check(False, "tokens and merge_mask must be on the same device")
    return merged


def co_me_token_split_cuda(merged_flat: torch.Tensor, rev_id: torch.Tensor, C: int) -> torch.Tensor:
    """Token split (inverse of merge): ``out[i, :] = merged_flat[rev_id[i], :]`` -> ``[total, C]``.
    ``rev_id`` may be int64 (as in the reference) or int32."""
    _torch_check(merged_flat.dim() == 2, "merged_flat must be [P, C]")
    return _lib.host().split(merged_flat, None, rev_id, C, [])


def co_me_token_split_pair_cuda(merged_a: torch.Tensor, merged_b: torch.Tensor, rev_id: torch.Tensor,
                                C: int) -> torch.Tensor:
    """Two token splits and the concatenation of their results in one launch:
    ``out[i] = cat(merged_a[rev_id[i]], merged_b[rev_id[i]])`` -> ``[total, 2 * C]``
    (the retained-layer step of the fused aggregator, reference ``vggt/fused.py:157-165``)."""
    return _lib.host().split(merged_a, merged_b, rev_id, C, [])


def co_me_token_merge_cuda_legacy(*args, **kwargs):
    """The reference still exports its first-generation pair (``co_me_cuext.pyi:22-46``) but calls it nowhere;
    it is not provided here."""
    raise RuntimeError("co_me_token_merge_cuda_legacy is not provided by the HIP build: use co_me_token_merge_cuda")


def co_me_token_merge_scan_legacy(*args, **kwargs):
    """See ``co_me_token_merge_cuda_legacy``."""
    raise RuntimeError("co_me_token_merge_scan_legacy is not provided by the HIP build: use co_me_token_merge_cuda")


def co_me_token_merge_2d_cuda(tokens: torch.Tensor, start_index: int, group_h: int, group_w: int, H: int, W: int,
                              merge_mask: torch.Tensor, index_dtype: torch.dtype = torch.int64,
                              count_dtype: torch.dtype = torch.float32):
    """2-D window merge straight from the image row-major token order (no permuted copy).

    ``tokens [B, start_index + H*W, C]``, ``merge_mask [B, (H//gh)*(W//gw)] bool``.  Grid positions
    outside the full windows are copied behind the windows.  Returns
    ``(out_flat [P,C], offsets [B+1] int32, index_map [B*N], counts [P])``.
    """
    _torch_check(tokens.is_cuda and merge_mask.is_cuda, "tokens and merge_mask must be on CUDA")
    _torch_check(tokens.dim() == 3 and merge_mask.dim() == 2, "tokens must be [B, N, C], merge_mask [B, M]")
    start_index, group_h, group_w, H, W = int(start_index), int(group_h), int(group_w), int(H), int(W)
    _torch_check(start_index >= 0 and group_h > 0 and group_w > 0 and H >= 0 and W >= 0, "bad geometry")
    B, N, _ = tokens.shape
    M = (H // group_h) * (W // group_w)
    _torch_check(merge_mask.shape[0] == B, "merge_mask batch != tokens batch")
    _torch_check(N == start_index + H * W, "N != start_index + H * W")
    _torch_check(merge_mask.shape[1] == M, "M != (H // group_h) * (W // group_w)")
    return _lib.host().merge_2d_flat(tokens, start_index, group_h, group_w, H, W, merge_mask.to(torch.bool),
                                     *_result_types(index_dtype, count_dtype), None)


def _result_types(index_dtype: torch.dtype, count_dtype: torch.dtype) -> tuple[bool, bool]:
    _torch_check(index_dtype in (torch.int64, torch.int32), "index_dtype must be int64 or int32")
    _torch_check(count_dtype in (torch.float32, torch.int32), "count_dtype must be float32 or int32")
    return index_dtype == torch.int64, count_dtype == torch.float32


_MODES = {"pairwise-rank": 0, "abs_mse": 1, "mse": 2}


def co_me_select_windows(conf: torch.Tensor, batch: int, group_h: int, group_w: int, threshold: float,
                         mode: str = "pairwise-rank", return_means: bool = False):
    """Window confidence means + lowest-confidence selection.

    ``conf [batch*frames, H, W]`` bf16 or fp32 -> ``mask [batch*frames, M] bool``
    (and the window means as float32 when ``return_means``).
    """
    _torch_check(conf.is_cuda, "conf must be on CUDA")
    _torch_check(conf.dim() == 3, "conf must be [B*S, H, W]")
    _torch_check(mode in _MODES, f"unsupported confidence mode {mode!r}")
    _torch_check(conf.dtype in (torch.bfloat16, torch.float32), "conf must be bfloat16 or float32")
    rows, H, W = conf.shape
    _torch_check(batch > 0 and rows % batch == 0, "conf rows must be a multiple of batch")
    lib = _lib.load()
    conf_c = conf.contiguous()
    dev = conf.device
    M = (H // group_h) * (W // group_w)
    with torch.cuda.device(dev):
        mask = torch.empty(rows, M, dtype=torch.bool, device=dev)
        means = torch.empty(rows, M, dtype=torch.float32, device=dev)
        _lib.check(lib.come_select_windows(conf_c.data_ptr(), _lib.dtype_code(conf_c.dtype), batch, rows // batch,
                                           H, W, group_h, group_w, _MODES[mode], float(threshold),
                                           means.data_ptr(), mask.data_ptr(), None, 0, _lib.current_stream(dev)))
    return (mask, means) if return_means else mask


def co_me_select_merge_2d(tokens: torch.Tensor, conf: torch.Tensor, batch: int, start_index: int, group_h: int,
                          group_w: int, H: int, W: int, ratio: float, index_dtype: torch.dtype = torch.int32,
                          count_dtype: torch.dtype = torch.int32, mode: str = "pairwise-rank"):
    """Confidence-guided merge in one call: window means -> joint lowest-``ratio`` selection per
    batch element -> merge plan (one launch for all three when ``batch == 1``) -> gather-mean.  Returns
    ``(merged [P,C], index_map [B_eff*N], counts [P], cu_seqlens [B_eff+1] int32, mask [B_eff,M] bool)``.
    """
    _torch_check(tokens.is_cuda and conf.is_cuda, "tokens and conf must be on CUDA")
    _torch_check(tokens.dim() == 3, "tokens must be [B, N, C]")
    _torch_check(mode in _MODES, f"unsupported confidence mode {mode!r}")
    _torch_check(conf.dtype in (torch.bfloat16, torch.float32), "conf must be bfloat16 or float32")
    start_index, group_h, group_w, H, W = int(start_index), int(group_h), int(group_w), int(H), int(W)
    _torch_check(start_index >= 0 and group_h > 0 and group_w > 0 and H >= 0 and W >= 0, "bad geometry")
    rows, N, _ = tokens.shape
    M = (H // group_h) * (W // group_w)
    _torch_check(N == start_index + H * W, "N != start_index + H * W")
    _torch_check(batch > 0 and rows % batch == 0, "token rows must be a multiple of batch")
    _torch_check(conf.numel() == rows * H * W, "conf must hold one value per grid position")
    if M == 0 or rows == 0:         # nothing to select from: every token is kept
        mask = torch.zeros(rows, M, dtype=torch.bool, device=tokens.device)
        out, offsets, index_map, counts = co_me_token_merge_2d_cuda(tokens, start_index, group_h, group_w, H, W, mask,
                                                                     index_dtype=index_dtype, count_dtype=count_dtype)
        return out, index_map, counts, offsets, mask
    mask, plan = _lib.host().select_plan(conf, batch, rows, H, W, group_h, group_w, float(ratio), _MODES[mode], start_index)
    out, offsets, index_map, counts = _lib.host().merge_2d_flat(tokens, start_index, group_h, group_w, H, W, mask,
                                                                *_result_types(index_dtype, count_dtype), plan)
    return out, index_map, counts, offsets, mask
