"""The GEMM tile configurations (256/128-row tiles of several widths, the small
tiles, split tail rows, paired launches) against the fp32-output kernel."""
import pytest
import torch

from tests.helpers import T128X96, T256, gemm_plan, pair_plan

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from ditserve_amd import ops

# rows at the edges of 64-, 128- and 256-row tiles and of one and several rounds of
# 256 workgroups; features off every tile width; K from a single 64-k stage (fewer
# stages than LDS buffers) to more stages than weight-prefetch batches
SHAPES = [(m, n, k) for n, k in ((1536, 64), (200, 192), (1544, 320), (4616, 128)) for m in (1, 127, 129, 1024, 2305)]
SHAPES += [(1560, 1536, 1536), (2048, 1536, 2048), (2560, 4608, 448), (1024, 8968, 256), (666, 6144, 576),
           (3480, 1536, 4160), (16416, 3072, 256), (4096, 1536, 4096),
           (1560, 4608, 1536), (666, 8960, 704), (5001, 3080, 64), (5001, 1544, 128), (1500, 4616, 192),
           (2500, 1544, 64), (1500, 1544, 192),
           (21000, 1536, 1536), (22000, 1536, 1536)]  # outputs of 62 MB, left in the caches, and 64 MB, stored past them


def _operands(m, n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    def r(*s):
        return torch.randn(s, generator=g, device="cuda")
    return r(m, k).bfloat16(), (r(n, k) * 0.05).bfloat16(), r(n), r(m, n).bfloat16(), r(2, n)


def _want(x, w, b, res, gate, seg, epi):
    """The epilogue in fp32 on the fp32-output kernel's products (whose sums the
    bf16 kernels share bit for bit)."""
    y = ops.linear(x, w, b, "f32").bfloat16()
    f = y.float()
    if epi == "bias":
        return y
    if epi == "gelu":
        return torch.nn.functional.gelu(f, approximate="tanh")
    if epi == "silu":
        return torch.nn.functional.silu(f)
    if epi == "res":
        return res.float() + f
    rows = torch.arange(x.shape[0], device="cuda") >= seg.cu[1]
    return res.float() + f * gate[rows.long()]


def _check(got, want, epi):
    if epi == "bias":
        assert torch.equal(got, want)
        return
    # one bf16 rounding of the result (2^-9 relative) and of the transcendentals' few fp32 ulps
    err = (got.float() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + 1e-5).all()), float(err.max())


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiles_match_the_fp32_output_kernel(m, n, k):
    x, w, b, res, gate = _operands(m, n, k, m + n + k)
    seg = ops.Segments([0, m // 3, m], "cuda")
    for epi in ("bias", "gelu", "silu", "res", "gate_res"):
        kw = dict(residual=res) if epi in ("res", "gate_res") else {}
        if epi == "gate_res":
            kw.update(gate=gate, segments=seg)
        out = torch.full((m + 1, n), 7.0, device="cuda", dtype=torch.bfloat16)
        ops.linear(x, w, b, epi, out=out[:m], **kw)
        _check(out[:m], _want(x, w, b, res, gate, seg, epi), epi)
        assert bool((out[m] == 7.0).all())  # nothing past the last row


# full rounds of 256 x 256 tiles, then the other rows on 128 x 96 ones (several tile rows
# at long K)
SPLITS = [(10914, 1536, 4096, 10752), (12001, 1536, 6144, 10752), (5505, 3072, 14336, 5376)]


@pytest.mark.parametrize("m,n,k,rows", SPLITS)
@pytest.mark.parametrize("epi", ["bias", "gelu", "res", "gate_res"])
def test_split_products(m, n, k, rows, epi):
    """A product in two launches, the second on gemm_kernel_l4 with a row base: against
    the fp32-output kernel, and bit for bit against the same rows as a product of
    their own.  The gated residual's segments end inside either part."""
    assert gemm_plan(m, n, k, epi) == (T256, rows, T128X96)
    x, w, b, res, gate = _operands(m, n, k, m + k)
    cut = [0, 4000, rows + 60, m]
    g = torch.randn((3, n), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")

    def run(lo, hi, out=None):
        kw = dict(residual=res[lo:hi]) if epi in ("res", "gate_res") else {}
        if epi == "gate_res":
            kw.update(gate=g, segments=ops.Segments([min(max(c - lo, 0), hi - lo) for c in cut], "cuda"))
        return ops.linear(x[lo:hi], w, b, epi, out=out, **kw)

    out = torch.full((m + 1, n), 7.0, device="cuda", dtype=torch.bfloat16)
    run(0, m, out[:m])
    assert bool((out[m] == 7.0).all())
    y = ops.linear(x, w, b, "f32").bfloat16()
    f = y.float()
    seg = torch.bucketize(torch.arange(m, device="cuda"), torch.tensor(cut[1:3], device="cuda"), right=True)
    want = {"bias": lambda: y, "gelu": lambda: torch.nn.functional.gelu(f, approximate="tanh"),
            "res": lambda: res.float() + f, "gate_res": lambda: res.float() + f * g[seg]}[epi]()
    _check(out[:m], want, epi)
    for lo, hi in ((rows, m), (rows - 200, rows + 100), (3900, 4100)):
        assert gemm_plan(hi - lo, n, k, epi)[0] != T256
        assert torch.equal(out[lo:hi], run(lo, hi)), (lo, hi)


@pytest.mark.parametrize("m", [1, 2, 15, 16])
@pytest.mark.parametrize("n,k", [(16384, 32), (16392, 96), (16440, 544), (20000, 1536)])
def test_few_rows_match_the_tiles(m, n, k):
    """Up to 16 rows run without LDS tiles: bit for bit the rows of a taller product."""
    x, w, b, res, gate = _operands(40, n, k, m + n + k)
    few, tall = ops.Segments([0, m // 2, m], "cuda"), ops.Segments([0, m // 2, 40], "cuda")
    for epi in ("f32", "bias", "gelu", "silu", "res", "gate_res"):
        kw = [dict(residual=res[:r]) if epi in ("res", "gate_res") else {} for r in (m, 40)]
        if epi == "gate_res":
            for d, seg in zip(kw, (few, tall)):
                d.update(gate=gate, segments=seg)
        out = torch.full((m + 1, n), 7.0, device="cuda", dtype=torch.float32 if epi == "f32" else torch.bfloat16)
        ops.linear(x[:m], w, b, epi, out=out[:m], **kw[0])
        assert torch.equal(out[:m], ops.linear(x, w, b, epi, **kw[1])[:m]), epi
        assert bool((out[m] == 7.0).all())
    y = x[:m].double() @ w.double().t() + b.double()
    assert float((ops.linear(x[:m], w, b, "f32").double() - y).norm() / y.norm()) < 1e-6  # fp32 sums of k products


@pytest.mark.parametrize("m0,m1,n,k", [(2048, 666, 1536, 6144), (2048, 666, 4608, 1536), (256, 100, 1536, 1536),
                                       (64, 2048, 1544, 64), (8192, 666, 1536, 256), (129, 1, 200, 128)])
@pytest.mark.parametrize("epi", ["bias", "gelu", "gate_res"])
def test_paired_tiles_match_single_launches(m0, m1, n, k, epi):
    probs = []
    for m, seed in ((m0, 1), (m1, 2)):
        x, w, b, res, gate = _operands(m, n, k, seed)
        p = dict(x=x, w=w, b=b)
        if epi == "gate_res":
            p.update(residual=res, gate=gate, segments=ops.Segments([0, m // 2, m], "cuda"))
        probs.append(p)
    assert pair_plan(m0, n, m1, n, k, epi) >= 0  # in one launch
    got = ops.linear_pair(*probs, epi)
    for g, p in zip(got, probs):
        assert torch.equal(g, ops.linear(epilogue=epi, **p))


@pytest.mark.parametrize("m0,n0,m1,n1,k", [(1560, 1536, 512, 3072, 1536), (2560, 1536, 1024, 3072, 1536),
                                           (77, 200, 1300, 1544, 64), (1300, 4616, 1, 8, 128)])
def test_paired_tiles_of_two_widths_match_single_launches(m0, n0, m1, n1, k):
    ps = [dict(zip("xwb", _operands(m, n, k, n + m)[:3])) for m, n in ((m0, n0), (m1, n1))]
    assert pair_plan(m0, n0, m1, n1, k) >= 0
    for g, p in zip(ops.linear_pair_n(*ps), ps):
        assert torch.equal(g, ops.linear(**p))
    with pytest.raises(ValueError, match="one N and K"):
        ops.linear_pair(*ps)
