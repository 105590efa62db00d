"""Dynamic Input Pruning (DIP) SwiGLU MLP for one decoder layer at batch 1.

Operation sequence of the reference's run_decoder_layer_dip /
run_decoder_layer_cached_dip MLP half (python/soinfer/runtime/generate.py:
276-310 and 367-404):

    gate  = INT4 GEMV(W_gate, x)                       dense, [I]
    idx   = topk_threshold_select(|gate| as fp32, k)   ascending indices
    u     = INT4 GEMV over rows idx of W_up            [k]
    h     = fp16(silu(fp32(gate[idx])) * fp32(u))      torch glue, as the reference
    y     = sum_j h_j * row idx_j of W_down^T          [H]

On MI355X all weights stay resident in HBM (288 GB), so the selected rows are
read in place through the index list (no host gather). dip_mlp_gathered runs
the reference's gather-then-GEMV shape on device buffers, and cached_dip_mlp
the hot-cache + staging shape; all three return bit-identical outputs for the
same inputs, because every path feeds the same kernel bodies the same
logical rows.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn.functional as F

from .. import _C
from .. import ops
from ..offload.hot_cache import HotCache


@dataclass
class DipMLPWeights:
    """INT4 g-group weights of one SwiGLU MLP. down is stored transposed ([I, H]) so that selecting
    intermediate channels is a row selection for both up and down (reference
    python/soinfer/offload/load_hf_checkpoint.py:90-111)."""

    gate_Wq: torch.Tensor  # [I, ceil(H/8)*4] uint8
    gate_scale: torch.Tensor  # [I, ceil(H/gs)] fp32
    up_Wq: torch.Tensor  # [I, ceil(H/8)*4]
    up_scale: torch.Tensor
    down_T_Wq: torch.Tensor  # [I, ceil(H/8)*4]
    down_T_scale: torch.Tensor  # [I, ceil(H/gs)]
    hidden_size: int
    group_size: int

    @property
    def intermediate_size(self) -> int:
        return int(self.gate_Wq.shape[0])


def select_channels(w: DipMLPWeights, x: torch.Tensor, dip_k: int) -> tuple[torch.Tensor, torch.Tensor]:
    """gate = W_gate x (dense) and the DIP selection idx (int32 [dip_k], ascending)."""
    gate, idx, _ = _C.dip_gate_select(w.gate_Wq, w.gate_scale, x, dip_k, w.hidden_size, w.group_size)
    return gate, idx


def silu_gate(gate: torch.Tensor, idx: torch.Tensor, u: torch.Tensor) -> torch.Tensor:
    """h_j = fp16(silu(fp32(gate[idx_j])) * fp32(u_j)) (generate.py:304-305)."""
    g_sel = gate.index_select(0, idx.long())
    return (F.silu(g_sel.float()) * u.float()).half()


def dip_mlp(w: DipMLPWeights, x: torch.Tensor, dip_k: int, channel_counts: Optional[torch.Tensor] = None):
    """Resident-weight DIP MLP. Returns (y [H] fp16, idx [dip_k] int32). Two launches: gate and up of every channel,
    then the selection inside the sparse down. up of an unselected channel is read and not used; leaving it out takes two
    launches more (top-k, and up over its selection: as cached_dip_mlp_direct), which cost more up to 4096 x 12288 (2048
    x 6144, k/I 0.05 / 0.3: 16.5 / 16.4 us against 23.7 / 22.6; 4096 x 12288: 25.9 / 29.5 against 25.4 / 30.2) and less
    where few of very many channels are selected (5120 x 17408: 38.3 / 43.4 against 34.1 / 43.2)."""
    count = None if channel_counts is None else torch.empty(1, dtype=torch.int32, device=x.device)
    y, idx = _C.dip_mlp(w.gate_Wq, w.gate_scale, w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, x, dip_k,
                        w.hidden_size, w.group_size, count)
    if channel_counts is not None:
        # fewer than k gates that are numbers: the list past the count is not written
        kept = torch.arange(idx.shape[0], dtype=torch.int32, device=idx.device) < count
        channel_counts.scatter_add_(0, torch.where(kept, idx, 0).long(), kept.to(channel_counts.dtype))
    return y, idx


def dip_mlp_gathered(w: DipMLPWeights, x: torch.Tensor, dip_k: int):
    """Reference-shaped DIP MLP: gather the selected up / down^T rows into compact buffers first, then
    gemv_w4a16_group_lop3 and gemv_w4a16_sparse_accumulate. Returns (y, idx)."""
    gate, idx = select_channels(w, x, dip_k)
    k = idx.shape[0]
    idx_l = idx.long()
    up_sel = torch.empty(k, w.up_Wq.shape[1], dtype=torch.uint8, device=x.device)
    down_sel = torch.empty(k, w.down_T_Wq.shape[1], dtype=torch.uint8, device=x.device)
    ops.gather_rows_device(w.up_Wq, idx, up_sel)
    ops.gather_rows_device(w.down_T_Wq, idx, down_sel)
    u = ops.gemv_w4a16_group_lop3(up_sel, w.up_scale.index_select(0, idx_l), x, w.hidden_size, w.group_size)
    h = silu_gate(gate, idx, u)
    y = ops.gemv_w4a16_sparse_accumulate(down_sel, w.down_T_scale.index_select(0, idx_l), h, w.hidden_size,
                                         w.group_size)
    return y, idx


def cached_dip_mlp(w: DipMLPWeights, cache: HotCache, x: torch.Tensor, dip_k: int,
                   host_up: Optional[torch.Tensor] = None, host_down_T: Optional[torch.Tensor] = None,
                   staging: Optional[torch.Tensor] = None, miss_bytes: Optional[list] = None):
    """Cache-aware DIP MLP: selected channels resident in `cache` are read from it, the misses from the
    device-resident weights (default) or, when host_up / host_down_T (pinned [I, row_nbytes]) and `staging` (pinned,
    >= dip_k * row_nbytes) are given, from pinned host memory. The kernels read pinned rows through their device
    mapping; host tensors that have none go through `staging` with the staged H2D gather. Bit-identical to dip_mlp.
    Returns (y, idx, miss_count)."""
    hosted = host_up is not None and host_down_T is not None
    if hosted and not _mapped(w, host_up, host_down_T, staging, dip_k):
        return _cached_mlp_staged(w, cache, x, dip_k, host_up, host_down_T, staging, miss_bytes)
    count = torch.empty(1, dtype=torch.int32, pin_memory=True)
    stream, read = torch.cuda.current_stream(x.device), torch.cuda.Event()
    try:
        gate, idx, ws = _C.dip_gate_select(w.gate_Wq, w.gate_scale, x, dip_k, w.hidden_size, w.group_size,
                                           cache.slot_of, count)
        if hosted:
            y = _cached_mlp(w, cache, x, gate, idx, ws, host_up, host_down_T, lambda: read.record(stream))
        else:
            read.record(stream)
            y = _cached_mlp(w, cache, x, gate, idx, ws, w.up_Wq, w.down_T_Wq)
    except BaseException:
        # what was launched before the failure still writes the count and reads the host rows: neither may be given
        # back before it has run
        stream.synchronize()
        raise
    # the count has arrived, and the host rows, which the caller may change or free once this returns, have been read
    read.synchronize()
    mc = int(count)
    if miss_bytes is not None:
        miss_bytes.append(mc * (w.up_Wq.shape[1] + w.down_T_Wq.shape[1]))
    return y, idx, mc


def _mapped(w: DipMLPWeights, host_up: torch.Tensor, host_down_T: torch.Tensor, staging, dip_k: int) -> bool:
    """Whether the host rows are pinned matrices of the weights' shapes (readable by the kernels), with the staging
    buffer that the gathers of the same call would need."""
    def pinned(t):
        return isinstance(t, torch.Tensor) and t.device.type == "cpu" and t.dtype == torch.uint8 and \
            t.is_contiguous() and t.is_pinned()

    return pinned(host_up) and pinned(host_down_T) and pinned(staging) and host_up.shape == w.up_Wq.shape and \
        host_down_T.shape == w.down_T_Wq.shape and \
        staging.numel() >= dip_k * max(host_up.shape[1], host_down_T.shape[1])


def _cached_mlp_staged(w: DipMLPWeights, cache: HotCache, x: torch.Tensor, dip_k: int, host_up, host_down_T, staging,
                       miss_bytes: Optional[list]):
    """cached_dip_mlp with the misses gathered on the host, one matrix after the other through `staging`."""
    gate, idx = select_channels(w, x, dip_k)
    desc, miss_channels, miss_count = ops.build_dip_descriptors(idx, cache.slot_of)
    mc = int(miss_count.item())
    miss_l = miss_channels[:mc].long()
    up_st = torch.empty(mc, w.up_Wq.shape[1], dtype=torch.uint8, device=x.device)
    down_st = torch.empty(mc, w.down_T_Wq.shape[1], dtype=torch.uint8, device=x.device)
    if mc:
        miss_cpu = miss_l.cpu()
        ops.gather_rows_staged(host_up, miss_cpu, staging, up_st)
        torch.cuda.current_stream().synchronize()  # staging reused for the second gather
        ops.gather_rows_staged(host_down_T, miss_cpu, staging, down_st)
    if miss_bytes is not None:
        miss_bytes.append(mc * (w.up_Wq.shape[1] + w.down_T_Wq.shape[1]))
    u = ops.gemv_dip_fused_up(cache.up_Wq, cache.up_scale, up_st, w.up_scale.index_select(0, miss_l), desc, x,
                              w.hidden_size, w.group_size)
    h = silu_gate(gate, idx, u)
    y = ops.gemv_dip_fused_down(cache.down_Wq, cache.down_scale, down_st, w.down_T_scale.index_select(0, miss_l), desc,
                                h, w.hidden_size, w.group_size)
    return y, idx, mc


def _cached_mlp(w: DipMLPWeights, cache: HotCache, x, gate, idx, ws, full_up, full_down_T,
                rows_read=lambda: None) -> torch.Tensor:
    """The up and down halves over the hot cache: hits from the cache, misses from full_up / full_down_T in place. For
    misses in host memory the up GEMV also copies its channels' down^T rows to the device (whole rows cross PCIe faster
    than the down's column slices). rows_read() is called after the last launch that reads full_up or full_down_T."""
    H, gs, k = w.hidden_size, w.group_size, idx.shape[0]
    h = torch.empty(k, dtype=torch.float16, device=x.device)
    row = full_down_T.shape[1]
    copy = not full_down_T.is_cuda and row % 16 == 0 and row <= 4096 and full_down_T.data_ptr() % 16 == 0
    staged = torch.empty(k, row, dtype=torch.uint8, device=x.device) if copy else None
    _C.gemv_dip_cached_up_silu_into(cache.up_Wq, cache.up_scale, full_up, w.up_scale, cache.slot_of, idx, x, gate, h, H,
                                    gs, full_down_T if copy else None, staged)
    if copy:
        rows_read()
    y = torch.empty(H, dtype=torch.float16, device=x.device)
    _C.gemv_dip_cached_down_into(cache.down_Wq, cache.down_scale, full_down_T, w.down_T_scale, cache.slot_of, idx, h, y,
                                 H, gs, ws, staged)
    if not copy:
        rows_read()
    return y


def cached_dip_mlp_direct(w: DipMLPWeights, cache: HotCache, x: torch.Tensor, dip_k: int,
                          full_up: Optional[torch.Tensor] = None, full_down_T: Optional[torch.Tensor] = None,
                          workspace: Optional[torch.Tensor] = None):
    """Cache-aware DIP MLP with the misses read in place: the up GEMV and the down accumulate resolve every
    selected channel through cache.slot_of themselves, reading hits from the cache and misses from full_up /
    full_down_T (pinned host memory read through its device mapping, or device tensors; default: the
    resident weights). No descriptors, no gather, no staging buffer and no host sync; the SiLU gating is the
    up GEMV's epilogue. Bit-identical to dip_mlp and cached_dip_mlp. Returns (y, idx)."""
    gate, idx, ws = _C.dip_gate_select(w.gate_Wq, w.gate_scale, x, dip_k, w.hidden_size, w.group_size)
    full_up = w.up_Wq if full_up is None else full_up
    full_down_T = w.down_T_Wq if full_down_T is None else full_down_T
    H, gs = w.hidden_size, w.group_size
    h = torch.empty(dip_k, dtype=torch.float16, device=x.device)
    _C.gemv_dip_cached_up_silu_into(cache.up_Wq, cache.up_scale, full_up, w.up_scale, cache.slot_of, idx, x, gate,
                                    h, H, gs)
    y = torch.empty(H, dtype=torch.float16, device=x.device)
    _C.gemv_dip_cached_down_into(cache.down_Wq, cache.down_scale, full_down_T, w.down_T_scale, cache.slot_of, idx,
                                 h, y, H, gs, ws if workspace is None else workspace)
    return y, idx


def calibrate_channel_frequencies(w: DipMLPWeights, xs: torch.Tensor, dip_k: int) -> torch.Tensor:
    """counts[c] = number of calibration inputs whose DIP selection contains channel c
    (generate.py:579-609, one layer). xs: [n, H] fp16."""
    counts = torch.zeros(w.intermediate_size, dtype=torch.int64, device=xs.device)
    for i in range(xs.shape[0]):
        dip_mlp(w, xs[i].contiguous(), dip_k, channel_counts=counts)
    return counts
