"""Attention outputs pinned bit for bit: the decisions of the lazy rescale (for 64
queries at a time) reach the rounding of every probability, so a change of them shows
in whole predictions.  The hashes were taken from the kernels with 256-query work items
only; launches of 128-query ones have to give the same."""
import hashlib
import json
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "attention_bits.json")
# heads, query and key rows per segment; small launches (128-query items) first
SHAPES = {
    "one": (3, [1560], [1560]),
    "cross": (12, [1280, 700], [512, 77]),
    "ragged": (3, [700, 31, 1290], [700, 31, 1290]),
    "short": (12, [300, 1, 90, 129], [300, 1, 90, 129]),
    "full": (24, [2600, 1357], [2600, 1357]),
}
JOINT = {"small": (4, [260, 64], [77, 33]), "pair": (24, [1024, 1024], [333, 154])}


def _rows(rng, rows, width, every, factor):
    """bf16 rows, every `every`-th scaled up so that running maxima rise past the rescale
    threshold for some queries of a wave and not for others."""
    x = rng.standard_normal((rows, width)).astype(np.float32)
    x[::every] *= factor
    return torch.from_numpy(x).to("cuda", torch.bfloat16)


def _cu(lens):
    return [0, *np.cumsum(lens).tolist()]


def _hash(*tensors):
    h = hashlib.sha256()
    for t in tensors:
        h.update(t.contiguous().view(torch.uint8).cpu().numpy().tobytes())
    return h.hexdigest()[:32]


def varlen_bits(name, d, pre):
    from ditserve_amd import ops
    heads, qlens, klens = SHAPES[name]
    rng = np.random.RandomState(len(name) + d + pre)
    q, k = _rows(rng, sum(qlens), heads * d, 37, 6.0), _rows(rng, sum(klens), heads * d, 53, 5.0)
    v = _rows(rng, sum(klens), heads * d, 1, 1.0)
    if pre:
        q = (q.float() * (d ** -0.5 * 1.4427)).bfloat16()
    return _hash(*ops.flash_attn_varlen(q, k, v, ops.Segments(_cu(qlens), "cuda"), ops.Segments(_cu(klens), "cuda"),
                                        heads, d, return_lse=True, q_prescaled=pre))


def joint_bits(name):
    from ditserve_amd import ops
    heads, img, txt = JOINT[name]
    rng = np.random.RandomState(7)
    w = heads * 64
    q, k = ([_rows(rng, sum(n), w, e, f) for n in (img, txt)] for e, f in ((37, 1.1), (53, 5.0)))
    v = [_rows(rng, sum(n), w, 1, 1.0) for n in (img, txt)]
    segs = [ops.Segments(_cu(n), "cuda") for n in (img, txt, [a + b for a, b in zip(img, txt)])]
    vt = ops.transpose_v_joint(*v, heads, 64, *segs)
    return _hash(*ops.joint_attention_q_prescaled(*q, *k, vt, *segs, heads, 64))


def all_bits():
    bits = {f"{n} d{d}{' pre' if pre else ''}": (varlen_bits, (n, d, pre))
            for n in SHAPES for d in (64, 128) for pre in (False, True)}
    bits.update({f"joint {n}": (joint_bits, (n,)) for n in JOINT})
    return bits


@pytest.mark.parametrize("case", list(all_bits()))
def test_attention_bits(case):
    fn, args = all_bits()[case]
    assert fn(*args) == json.load(open(GOLDEN))[case]
