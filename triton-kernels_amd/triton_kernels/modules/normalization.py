"""RMSNorm / QKNorm modules on the HIP rms_norm (modules/normalization.py:8-26 of the reference).
Parameter names (`scale`, `query_norm`, `key_norm`) are part of the state-dict contract."""
import torch
from torch import Tensor, nn
from torch.nn.modules.module import _has_any_global_hook

from triton_kernels.kernels.normalization import rms_norm, rms_norm_pair


def plain(module: nn.Module, cls: type) -> bool:
    """Whether calling `module` does what `cls` does and nothing else, so that its weights may be used directly."""
    return (type(module) is cls and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or _has_any_global_hook()))


class RMSNorm(nn.Module):
    def __init__(self, dim: int) -> None:
        super().__init__()
        self.scale = nn.Parameter(torch.ones(dim))

    def forward(self, x: Tensor) -> Tensor:
        return rms_norm(x, self.scale)


class QKNorm(nn.Module):
    def __init__(self, dim: int) -> None:
        super().__init__()
        self.query_norm = RMSNorm(dim)
        self.key_norm = RMSNorm(dim)

    def forward(self, q: Tensor, k: Tensor, v: Tensor) -> tuple[Tensor, Tensor]:
        if plain(self.query_norm, RMSNorm) and plain(self.key_norm, RMSNorm) and not torch.is_grad_enabled():
            q, k = rms_norm_pair(q, self.query_norm.scale, k, self.key_norm.scale)
            return q.to(v), k.to(v)
        return self.query_norm(q).to(v), self.key_norm(k).to(v)
