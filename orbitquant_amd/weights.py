"""Offline (host, torch) weight quantization: the tensors the packed GEMM reads.

Per output row (src/orbitquant/layers.py:121-125,201-215): `r = ||W_row||` in
fp32 on the unrotated row, `rotW = RPBH(W_row)`, `unit = rotW / max(r, eps)`,
`idx = #{j : boundaries[j] < unit}`, indices bit-packed as one flat little-endian
stream over the [N, K] index matrix, `row_norms = bf16(r)`.  A zero row keeps
`r = 0` and therefore dequantizes to exact zeros.

A weight that already sits on the GPU is quantized there (`oq_quantize_weight`, the
counterpart of the reference's device-side path, src/orbitquant/layers.py:102-125 with
src/orbitquant/kernels/triton_cuda.py:926-1039); a host weight takes the torch path below.
The two differ in one place only: the GPU kernel sums the squares of a row in the fixed order
of the activation kernel, the host path in torch's, so an index can differ where the last bit of
a norm moves a value across a boundary it sits on (the reference's own host and device paths
differ in the same way).
"""

from __future__ import annotations

import torch

from .codebooks import LloydMaxCodebook
from .packing import pack_lowbit
from .rotations import RPBHRotation


def quantize_weight_indices(
    weight: torch.Tensor,
    row_norms: torch.Tensor,
    *,
    rotation: RPBHRotation,
    codebook: LloydMaxCodebook,
    eps: float,
) -> torch.Tensor:
    rotated = rotation.apply_to_weight(weight)
    unit = rotated / row_norms.clamp_min(eps)[:, None]
    return codebook.quantize_indices(unit)


def quantized_on_gpu(weight: torch.Tensor, rotation: RPBHRotation) -> bool:
    """Whether the GPU's quantizer takes this weight."""
    k = weight.shape[1]
    return (weight.device.type == "cuda" and k % 8 == 0 and k <= 16384 and 8 <= rotation.block_size <= 4096
            and weight.dtype in (torch.float32, torch.float16, torch.bfloat16))


def quantize_weight(
    weight: torch.Tensor,
    *,
    rotation: RPBHRotation,
    codebook: LloydMaxCodebook,
    bits: int,
    eps: float,
    row_tile: int = 4096,
    constants: tuple[torch.Tensor, torch.Tensor, torch.Tensor] | None = None,
    plan: torch.Tensor | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """-> (packed uint8 [ceil(N*K*bits/8)], row_norms bfloat16 [N]), on the GPU for a GPU weight the
    kernel takes, else on the CPU.  `row_tile` bounds the rows whose fp32 copies the host path holds at a
    time; the result does not depend on it, and a GPU weight is one launch without such copies.
    `constants`: permutation (int32), signs (int8) and boundaries where they are on the weight's device already, and
    `plan` the rotate plan of these."""
    if weight.ndim != 2:
        raise ValueError("weight must be a matrix")
    n, k = weight.shape
    if quantized_on_gpu(weight, rotation):
        from . import ops

        device = weight.device
        # (one launch for the matrix: at 256 rows a launch, one workgroup a CU, 14336 x 4096 took 56 launches of 16 us
        # and some 200 us of Python; one launch 80 us)
        if constants is None:
            constants = (rotation.permutation.to(torch.int32).to(device), rotation.signs.to(torch.int8).to(device),
                         codebook.boundaries.to(device))
        return ops.quantize_weight(
            weight, *constants, bits=bits, block_size=rotation.block_size, eps=eps,
            inv_sqrt_block=rotation.normalization, plan=plan)
    # Tiles must end on a byte boundary of the flat stream: rows * k * bits % 8 == 0.
    align = 8
    while (align // 2) * k * bits % 8 == 0 and align > 1:
        align //= 2
    row_tile = max(align, row_tile // align * align)
    pieces: list[torch.Tensor] = []
    norms = torch.empty(n, dtype=torch.bfloat16)
    for start in range(0, n, row_tile):
        tile = weight[start : start + row_tile].detach().to(device="cpu", dtype=torch.float32)
        r = tile.norm(dim=-1)
        idx = quantize_weight_indices(tile, r, rotation=rotation, codebook=codebook, eps=eps)
        pieces.append(pack_lowbit(idx, bits, validate=False))
        norms[start : start + row_tile] = r.to(torch.bfloat16)
    return torch.cat(pieces), norms
