"""Shared helpers for the parity tests: error metric, seeded inputs built on the CPU (so every box reproduces them),
and oracle-side views of GPU-produced weights."""
import numpy as np
import torch

from oracle import quant_ref as Q

DEV = "cuda"


def err(out, ref):
    """(max_abs, max_rel) with max_rel = max_abs / max|ref| — normwise, as tests/test_kernels.py:30-38."""
    out, ref = out.detach().float().cpu(), ref.detach().float().cpu()
    max_abs = (out - ref).abs().max().item() if out.numel() else 0.0
    return max_abs, max_abs / max(ref.abs().max().item(), 1e-12)


def assert_close(out, ref, tol, what=""):
    max_abs, max_rel = err(out, ref)
    assert np.isfinite(max_abs) and max_rel <= tol, f"{what}: max_abs={max_abs:.3e} max_rel={max_rel:.3e} tol={tol}"
    return max_rel


def gen(seed):
    return torch.Generator().manual_seed(seed)


def make_cache(ctx, n_kv, page, D=64, peaky=1.0, seed=0, extra_pages=3):
    """Paged caches with a random block table over ctx/page + extra pages (tests/test_kernels.py:90-95)."""
    g = gen(seed)
    n_pages = (ctx + page - 1) // page + extra_pages
    kc = (torch.randn(n_pages, n_kv, page, D, generator=g) * peaky).half()
    vc = torch.randn(n_pages, n_kv, page, D, generator=g).half()
    bt = torch.randperm(n_pages, generator=g).int()
    return kc, vc, bt


def dequant_from_gpu(packed, sz, group):
    """fp16 w_ref [N, K] from GPU-produced packed / sz, through the oracle's unpack + dequantize."""
    q = Q.unpack(packed.cpu().numpy())
    s, z = Q.unpack_scale_zero(sz.cpu().numpy())
    return torch.from_numpy(Q.dequantize(q, s, z, group))


# (kernel, M, N, K, epilogue, splits) at G 128: every tiling of the register-stationary kernel and of the few-token one,
# with odd and even numbers of 128-wide chunks (three and more, so that its two-chunk pipeline turns over), 16-byte rows and
# rows that take element-wise stores (N % 4 != 0), both epilogues, and k ranges of equal and unequal lengths
GEMM_TILING_CASES = [
    ("rs 512x128 w8", 451, 24656, 896, 1, 1), ("rs 512x128 w8", 389, 28160, 1024, 0, 1),
    ("rs 512x128 w8", 450, 24786, 1024, 1, 1), ("rs 512x128 w8", 194, 8656, 8320, 0, 4),
    ("rs 512x128 w8", 194, 16656, 8192, 0, 2),
    ("rs 256x128 w8", 194, 24640, 384, 1, 1), ("rs 256x128 w8", 193, 16624, 512, 0, 1),
    ("rs 256x128 w8", 194, 24702, 896, 0, 1), ("rs 256x128 w8", 136, 5616, 8960, 0, 4),
    ("rs 256x128 w8", 775, 2464, 8192, 0, 2),
    ("rs 256x64 w8", 65, 16624, 384, 1, 1), ("rs 256x64 w8", 65, 16496, 512, 0, 1), ("rs 256x64 w8", 66, 16590, 384, 1, 1),
    ("rs 256x64 w8", 65, 1040, 14464, 0, 16), ("rs 256x64 w8", 65, 4368, 8320, 0, 4),
    ("rs 256x128 w4", 393, 28032, 384, 0, 1), ("rs 256x128 w4", 389, 27984, 512, 1, 1),
    ("rs 256x128 w4", 395, 27936, 384, 1, 1), ("rs 256x128 w4", 519, 21906, 384, 1, 1),
    ("rs 256x128 w4", 583, 23081, 512, 0, 1), ("rs 256x128 w4", 262, 21632, 8320, 0, 2),
    ("rs 128x128 w4", 326, 10848, 384, 0, 1), ("rs 128x128 w4", 341, 10848, 512, 1, 1),
    ("rs 128x128 w4", 193, 25150, 384, 1, 1), ("rs 128x128 w4", 1236, 4890, 896, 0, 1),
    ("rs 128x128 w4", 1748, 272, 8960, 0, 4), ("rs 128x128 w4", 1969, 592, 4224, 0, 2),
    ("rs 128x64 w4", 65, 10160, 384, 0, 1), ("rs 128x64 w4", 65, 10128, 512, 1, 1), ("rs 128x64 w4", 65, 10202, 384, 0, 1),
    ("rs 128x64 w4", 67, 464, 14464, 0, 16), ("rs 128x64 w4", 819, 272, 4224, 0, 2), ("rs 128x64 w4", 77, 912, 8320, 0, 8),
    ("rs 128x64 w4 few", 33, 20384, 384, 0, 1), ("rs 128x64 w4 few", 33, 20386, 512, 1, 1),
    ("rs 128x64 w4 few", 33, 20711, 512, 0, 1), ("rs 128x64 w4 few", 33, 1008, 14464, 0, 16),
    ("rs 128x64 w4 few", 34, 1984, 8320, 0, 8),
    ("thin 128", 16, 20480, 1152, 1, 1), ("thin 128", 32, 20486, 1024, 0, 1), ("thin 128", 32, 4100, 14336, 0, 8),
    ("thin 64", 9, 10250, 1280, 1, 1), ("thin 32", 32, 4992, 1152, 0, 1), ("thin 16", 17, 4096, 1408, 1, 1)]
