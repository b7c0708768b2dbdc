"""The attention plugin on [B, H, S, D] operands read in place, against the packed
entry point on packed copies (the same kernel, so bit for bit)."""
import pytest
import torch

from tests.helpers import attn_items

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from ditserve_amd import attention, ops


def _views(b, h, s, d, g):
    """Named [b, h, s, d] views of random memory: in place and not."""
    def r(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()
    yield "bhsd", r(b, h, s, d)
    yield "bshd", r(b, s, h, d).transpose(1, 2)
    yield "sbhd", r(s, b, h, d).permute(1, 2, 0, 3)
    yield "column slice", r(b, s, h, 3 * d).transpose(1, 2)[..., d:2 * d]
    yield "row slice", r(b, h, s + 5, d)[:, :, 3:s + 3]
    yield "shared batch", r(1, h, s, d).expand(b, h, s, d)
    yield "shared row", r(b, h, 1, d).expand(b, h, s, d)     # row stride 0
    yield "odd strides", r(b, h, s, d + 1)[..., :d]          # rows not 16-byte aligned: copied
    yield "dim stride", r(b, h, d, s).transpose(2, 3)        # D not contiguous: copied


@pytest.mark.parametrize("b,h,sq,sk,d", [(1, 3, 260, 260, 128), (2, 2, 77, 513, 128), (3, 2, 129, 64, 64),
                                         (2, 1, 1, 1, 64), (1, 24, 1357, 1357, 64), (2, 2, 40, 0, 128)])
def test_strided_operands_match_packed(b, h, sq, sk, d):
    g = torch.Generator(device="cuda").manual_seed(sq + sk + d)
    qs, ks, vs = (list(_views(b, h, s, d, g)) for s in (sq, sk, sk))
    seg_q, seg_k = ops.Segments.uniform(b, sq, "cuda"), ops.Segments.uniform(b, sk, "cuda")

    def rows(x):
        return x.transpose(1, 2).reshape(-1, h * d).contiguous()
    # each layout of q with another layout of k and of v
    for i, (name, q) in enumerate(qs):
        k, v = ks[(i + 3) % len(ks)][1], vs[(i + 5) % len(vs)][1]
        out, lse = attention.ditk_attention(q, k, v)
        want, want_lse = ops.flash_attn_varlen(rows(q), rows(k), rows(v), seg_q, seg_k, h, d, return_lse=True)
        assert out.shape == (b, h, sq, d) and lse.shape == (b, h, sq), name
        assert torch.equal(out, want.view(b, sq, h, d).transpose(1, 2)), name
        assert torch.equal(lse, want_lse.view(h, b, sq).permute(1, 0, 2)), name


def _spiky(t, h, d, seed):
    """q, k with occasional large rows, so that running maxima rise past the lazy
    rescale threshold for some queries of a wave and not for others."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn((t, h * d), generator=g, device="cuda") for _ in range(3))
    q[::37] *= 6.0
    k[::53] *= 5.0
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("pre", [False, True])
@pytest.mark.parametrize("lens", [[1, 64, 65], [127, 128, 129, 257], [700, 31, 1290], [1560], [0, 300, 5]])
def test_work_item_size_does_not_change_results(d, pre, lens):
    """A few short segments run as 128-query work items; the same segments packed
    with enough others to fill the GPU run as 256-query ones: bit for bit the same,
    rescales and lse included, and each close to softmax attention in fp64."""
    h, total = 3, sum(lens)
    assert attn_items(total, total, len(lens), h) == 128
    q, k, v = _spiky(total, h, d, total + d)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    seg = ops.Segments(cu, "cuda")
    few, few_lse = ops.flash_attn_varlen(q, k, v, seg, seg, h, d, return_lse=True, q_prescaled=pre)
    reps = 256 * 256 // max(total, 1) + 2
    cu_many = [0] + [r * total + c for r in range(reps) for c in cu[1:]]
    seg_many = ops.Segments(cu_many, "cuda")
    assert attn_items(reps * total, reps * total, reps * len(lens), h) == 256
    many, many_lse = ops.flash_attn_varlen(q.repeat(reps, 1), k.repeat(reps, 1), v.repeat(reps, 1), seg_many, seg_many,
                                           h, d, return_lse=True, q_prescaled=pre)
    for r in (0, reps // 2, reps - 1):
        assert torch.equal(many[r * total:(r + 1) * total], few)
        assert torch.equal(many_lse[:, r * total:(r + 1) * total], few_lse)
    scale = (1.0 / ops.LOG2E) if pre else d ** -0.5
    for a, b in zip(cu, cu[1:]):
        if a == b:
            continue
        qs, ks, vs = (x[a:b].double().view(b - a, h, d).transpose(0, 1) for x in (q, k, v))
        s = qs @ ks.transpose(1, 2) * scale
        want = (s.softmax(-1) @ vs).transpose(0, 1).reshape(b - a, h * d)
        err = (few[a:b].double() - want).norm() / want.norm()
        # P and O round to bf16 (2^-9 each, averaged over keys)
        assert float(err) < 8e-3, float(err)
        assert torch.allclose(few_lse[:, a:b].double(), s.logsumexp(-1), atol=2e-3, rtol=1e-5)



@pytest.mark.parametrize("img,txt", [([260, 64], [77, 33]), ([1], [63]), ([64, 129, 300], [64, 1, 20]), ([1024], [333])])
def test_joint_work_item_size_does_not_change_results(img, txt):
    """Joint attention likewise: segments whose last key tile is partial, whose image
    and text rows meet inside a tile or at its edge, on the one- and the two-block body,
    each close to softmax attention in fp64."""
    h, w = 4, 4 * 64
    def cu(lens, reps=1):
        out = [0]
        for n in lens * reps:
            out.append(out[-1] + n)
        return out
    both = [a + b for a, b in zip(img, txt)]
    total = sum(both)
    q, k, v = (dict(zip(("img", "txt"), x.split([sum(img), sum(txt)]))) for x in _spiky(total, w // 64, 64, total))
    q = {n: (x.float() * (64 ** -0.5 * ops.LOG2E)).bfloat16() for n, x in q.items()}

    def run(reps):
        segs = [ops.Segments(cu(n, reps), "cuda") for n in (img, txt, both)]
        (qi, qt), (ki, kt), (vi, vt_) = ([x[n].repeat(reps, 1) for n in ("img", "txt")] for x in (q, k, v))
        vt = ops.transpose_v_joint(vi, vt_, h, 64, *segs)
        return ops.joint_attention_q_prescaled(qi, qt, ki, kt, vt, *segs, h, 64)
    reps = 256 * 128 // total + 2
    assert attn_items(total, total, len(img), h, joint=True) == 128
    assert attn_items(reps * total, reps * total, reps * len(img), h, joint=True) == 256
    few, many = run(1), run(reps)
    for one, all_ in zip(few, many):
        for r in (0, reps // 2, reps - 1):
            assert torch.equal(all_[r * one.shape[0]:(r + 1) * one.shape[0]], one)
    for m in range(len(img)):
        rows = [slice(cu(n)[m], cu(n)[m + 1]) for n in (img, txt)]
        qs, ks, vs = (torch.cat([x[n][r] for n, r in zip(("img", "txt"), rows)]).double().view(-1, h, 64).transpose(0, 1)
                      for x in (q, k, v))
        want = ((qs @ ks.transpose(1, 2) / ops.LOG2E).softmax(-1) @ vs).transpose(0, 1).reshape(-1, w)
        got = torch.cat([x[r] for x, r in zip(few, rows)]).double()
        # P and O round to bf16 (2^-9 each, averaged over keys)
        assert float((got - want).norm() / want.norm()) < 8e-3
