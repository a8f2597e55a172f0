"""Host wrappers of the normalisation / rotary / gated-activation kernels (C ABI: kvx_rmsnorm_rows,
kvx_add_rmsnorm_rows, kvx_swiglu_rows, kvx_qk_norm_rope)."""
from typing import Optional, Tuple

import torch

from keys_values_amd import _lib


def rope_tables(context: int, head_size: int, base: float, device) -> Tuple[torch.Tensor, torch.Tensor]:
    """fp32 cos / sin tables (context, head_size / 2): row p holds cos / sin of p * base^(-2j / head_size).
    Half-split convention: element d of a head is paired with d +- head_size / 2
    (keys_values/fused/fused_rope.py:57-87,198-200)."""
    inv = 1.0 / (base ** (torch.arange(0, head_size, 2, dtype=torch.float32, device=device) / head_size))
    ang = torch.arange(context, dtype=torch.float32, device=device).unsqueeze(-1) * inv
    return ang.cos().contiguous(), ang.sin().contiguous()


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """RMSNorm.forward over the last axis (keys_values/model.py:870-878). x bf16 (..., dim), rows contiguous."""
    return _lib.host().rmsnorm(x, weight, eps, out)


def add_rmsnorm_(x: torch.Tensor, delta: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """``x += delta`` (in place, rounded to bf16) and ``RMSNorm(x)`` in one pass: the residual add of a
    block with the normalisation that follows it (keys_values/model.py:560-584). Returns the normed rows."""
    return _lib.host().add_rmsnorm(x, delta, weight, eps)


def swiglu(gate_up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` for ``gate_up = [gate | up]`` (..., 2 * dim), the output of one GEMM over the
    stacked fc_1 / fc_2 weights; same rounding as ``F.silu(gate) * up`` on bf16 tensors."""
    return _lib.host().swiglu(gate_up)


def qk_norm_rope_(qkv: torch.Tensor, n_head: int, n_query_groups: int, head_size: int, q_weight: Optional[torch.Tensor],
                  k_weight: Optional[torch.Tensor], eps: float, cos: torch.Tensor, sin: torch.Tensor, input_pos: int) -> torch.Tensor:
    """In place on qkv (B, num, (n_head + 2 n_query_groups) * head_size): norm_q / norm_k over each
    head and the rotary encoding at positions input_pos .. input_pos + num - 1
    (keys_values/model.py:733-775). Returns qkv."""
    _lib.host().qk_norm_rope(qkv, n_head, n_query_groups, head_size, q_weight, k_weight, eps, cos, sin, input_pos)
    return qkv
