"""Shared numerics helpers for the parity tests."""
import torch


def bf(x):
    """Round to bf16 values (kept as fp32): the inputs both sides see."""
    return x.to(torch.bfloat16).float()


def metrics(got, ref):
    """(cosine, relative L2, max abs err) of got vs ref, in float64."""
    g = got.double().reshape(-1).cpu()
    r = ref.double().reshape(-1).cpu()
    cos = float(torch.nn.functional.cosine_similarity(g, r, dim=0))
    rel = float((g - r).norm() / r.norm().clamp_min(1e-30))
    return cos, rel, float((g - r).abs().max())


def assert_close(got, ref, cos_min=0.999, rel_max=1e-2, label=""):
    cos, rel, mx = metrics(got, ref)
    assert torch.isfinite(got.float()).all(), f"{label}: non-finite output"
    assert cos >= cos_min and rel <= rel_max, f"{label}: cos={cos:.6f} relL2={rel:.3e} maxabs={mx:.3e}"
    return cos, rel


def gen(seed):
    return torch.Generator().manual_seed(seed)


def randn(shape, seed, scale=1.0):
    return torch.randn(shape, generator=gen(seed)) * scale


# Tiles of a product, as numbered by ditk_gemm_plan (2-7: one wave per SIMD)
SMALL, EIGHT_WAVES, T256, T128X192, T128X96, SKINNY = 0, 1, 2, 5, 7, 8


def gemm_plan(m, n, k, epi="bias"):
    """(tile, rows, rest tile) ditk_gemm takes for an m x n x k product: host only."""
    import ctypes

    from ditserve_amd import _lib, ops
    plan = (ctypes.c_int * 3)()
    _lib.call("ditk_gemm_plan", m, n, k, ops.EPILOGUES[epi], plan)
    return tuple(plan)


def pair_plan(m0, n0, m1, n1, k, epi="bias"):
    """The tile of a pair's one launch, -1 for two launches."""
    from ditserve_amd import _lib, ops
    return _lib.load().ditk_gemm_pair_plan(m0, n0, m1, n1, k, ops.EPILOGUES[epi])


def attn_items(tq, tk, nseg, heads, equal=False, joint=False):
    """Queries per work item (128 or 256) of an attention launch: host only."""
    from ditserve_amd import _lib
    return _lib.load().ditk_attn_item_queries(tq, tk, nseg, heads, equal, joint)
