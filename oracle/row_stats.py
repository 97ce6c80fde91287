"""Row statistics of a bf16 matrix in the order in which an encoder's first block takes them (fp32 additions one by one)."""

from __future__ import annotations

import torch


def in_chunk_order(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """fp32 [rows, 8] sums of squares and sums of 160-column parts of bf16 `x` (at most 1280 columns, a multiple of 8).

    A chunk of 8 columns is summed from left to right, starting at zero (the square of a bf16 value is exact in fp32, so a
    fused multiply-add rounds as the addition does).  Chunks c, c + 64 and c + 128 belong to lane c; a lane adds its chunks
    of a part in that order, and the 64 lanes meet in a tree: 32 apart, then 16, 8, 4, 2, 1."""
    rows, H = x.shape
    v = torch.zeros((rows, 3 * 64 * 8), dtype=torch.float32)
    v[:, :H] = x.float()
    v = v.view(rows, 3, 64, 8)
    out = []
    for terms in (v * v, v):
        chunk = torch.zeros((rows, 3, 64))
        for e in range(8):
            chunk = chunk + terms[..., e]
        lanes = torch.zeros((rows, 64, 8))
        for j in range(3):
            part = (torch.arange(64) + 64 * j) // 20
            for q in range(8):
                lanes[:, part == q, q] += chunk[:, j, part == q]
        while lanes.shape[1] > 1:
            half = lanes.shape[1] // 2
            lanes = lanes[:, :half] + lanes[:, half:]
        out.append(lanes[:, 0].contiguous())
    return out[0], out[1]
