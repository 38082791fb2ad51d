"""Which kernel serves a batched 3-bit product (for tests, which state what they run)."""
import hecbench_amd
from hecbench_amd import _lib


def kernel_of(M, K, N):
    """By the choice that the launch makes, with the present knobs, on the current device: "block" (the matvec's kernel, four rows
    side by side), "direct" (one launch), "rows64" (64 rows at a time behind a pre-pass) or "tiles" (many rows)."""
    choose = getattr(_lib.load(), "_Z18hq_q3_batch_kerneliiii")  # HqQ3Kernel of csrc/hq_internal.h
    return ("block", "direct", "rows64", "tiles")[choose(hecbench_amd.device_info()["compute_units"], K, N, M)]
