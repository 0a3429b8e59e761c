"""Pairs in the order that the grouped expert product takes, by torch operations."""

import torch


def sort_pairs_by_expert(selected: torch.Tensor, num_experts: int, rows: int):
    """Expert-sorted (token, slot) pair ids, each expert's segment padded to a multiple of `rows`:
    (sorted_pairs [Rp] i32 with -1 padding, tile_expert [Rp / rows] i32), Rp the most there can be."""
    dev = selected.device
    sel = selected.reshape(-1)  # [R] expert per pair
    R = sel.shape[0]
    order = torch.argsort(sel, stable=True)
    sel_sorted = sel[order]
    counts = torch.bincount(sel, minlength=num_experts)
    padded = (counts + rows - 1) // rows * rows
    pad_off = torch.cumsum(padded, 0) - padded       # padded segment starts
    unpad_off = torch.cumsum(counts, 0) - counts     # unpadded segment starts
    slot = pad_off[sel_sorted] + (torch.arange(R, device=dev) - unpad_off[sel_sorted])
    rp = (R + num_experts * (rows - 1) + rows - 1) // rows * rows  # static upper bound
    sorted_pairs = torch.full((rp,), -1, dtype=torch.int32, device=dev)
    sorted_pairs[slot] = order.to(torch.int32)
    tile_expert = torch.full((rp // rows,), -1, dtype=torch.int32, device=dev)
    tile_expert[slot // rows] = sel_sorted.to(torch.int32)
    return sorted_pairs, tile_expert
