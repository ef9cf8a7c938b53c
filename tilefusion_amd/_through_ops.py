"""What `_direct` is where that extension module is not built for the running interpreter: no call is taken, and the wrappers
of tilefusion_amd.ops go through torch.ops (about 1 us more a call)."""

from typing import Any


def gemm(*args: Any) -> bool:
    return False


def fused_two_gemms(*args: Any) -> bool:
    return False


def scatter_nd(*args: Any) -> bool:
    return False


def flash_attention(*args: Any) -> None:
    return None


def flash_decode(*args: Any) -> None:
    return None
