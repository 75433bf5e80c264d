"""The float32 paged decode kernel (f32 matrix instructions) against 64-bit
softmax attention: tile edges (16 tokens a tile, 64 tokens a page lookup, four
waves a workgroup), one split and several, GQA groups of 1 to 16, head_dim 64
and 128, pages of 1 to 48 tokens, an empty sequence, page ids outside the pool,
NaN in slots past a sequence's end, strided caches; and the call without a
workspace, which computes the same splits in one workgroup: bit-identical.
Tolerance: an output is a mean of V rows of order 1 in 32-bit sums, 1e-5
(about 1e-6 is measured)."""

import pytest
import torch

from tests.helpers import assert_bitexact
from tinyserver_amd import _lib
from tinyserver_amd.kernels import paged_attention_forward

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(lens, hq, hkv, d, page, seed):
    g = torch.Generator().manual_seed(seed)
    need = [max(1, -(-n // page)) for n in lens]
    pages = sum(need) + 3
    kc, vc = (torch.randn(pages, hkv, page, d, generator=g) for _ in range(2))
    perm, bt, at = torch.randperm(pages, generator=g), torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for s, n in enumerate(need):
        bt[s, :n] = perm[at:at + n]
        at += n
    return torch.randn(len(lens), hq, d, generator=g), kc, vc, bt, torch.tensor(lens, dtype=torch.int32)


def _exact(q, kc, vc, bt, lens):
    out = torch.full(q.shape, float("nan"), dtype=torch.float64)
    page, group = kc.shape[2], q.shape[1] // kc.shape[1]
    for s, n in enumerate(lens):
        pos = [(int(bt[s, t // page]), t % page) for t in range(n)]
        pos = [(p, i) for p, i in pos if 0 <= p < kc.shape[0]]
        if not pos:
            continue
        pg, sl = (torch.tensor(x) for x in zip(*pos))
        for h in range(q.shape[1]):
            k, v = kc[pg, h // group, sl].double(), vc[pg, h // group, sl].double()
            out[s, h] = torch.softmax(k @ q[s, h].double() * q.shape[2] ** -0.5, 0) @ v
    return out


def _noalloc(q, kc, vc, bt, sl):
    out = torch.empty_like(q)
    views = [_lib.view(t) for t in (out, q, kc, vc, bt, sl)]
    _lib.check(_lib.load().tsa_paged_decode_noalloc(*map(_lib.ref, views), q.shape[-1] ** -0.5, 0,
                                                    torch.cuda.current_stream().cuda_stream), "noalloc")
    return out


@pytest.mark.parametrize("hq,hkv,d,page,lens", [
    (16, 8, 128, 4, [1, 15, 16, 17, 64, 65, 127, 1000]),  # several splits
    (4, 2, 128, 16, [0, 5, 300, 512]),                    # one split
    (3, 3, 64, 1, [1, 33, 600, 2]),
    (32, 2, 128, 48, [700, 47, 49, 2500]),
    (10, 2, 64, 7, [6, 7, 8, 1111]),
    (8, 8, 128, 256, [255, 257, 4096, 1] * 20),           # 640 units
])
def test_against_64_bits(hq, hkv, d, page, lens):
    q, kc, vc, bt, sl = _inputs(lens, hq, hkv, d, page, seed=d + page)
    ref = _exact(q, kc, vc, bt, lens)
    for s, n in enumerate(lens):  # what lies past a sequence's end must not be read
        if n % page:
            kc[bt[s, n // page], :, n % page:] = float("nan")
            vc[bt[s, n // page], :, n % page:] = float("inf")
    args = [t.to(DEV) for t in (q, kc, vc, bt)]
    out = paged_attention_forward(*args, page, sl.to(DEV))
    assert_bitexact(_noalloc(*args, sl.to(DEV)), out, "without a workspace")
    out = out.cpu().double()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    err = float((out - ref).nan_to_num().abs().max())
    print(f"{hq}/{hkv} x {d}, page {page}: max_abs={err:.2e}", flush=True)
    assert err <= 1e-5


def test_page_ids_outside_the_pool():
    q, kc, vc, bt, sl = _inputs([100, 900], 4, 2, 128, 16, seed=3)
    bt[0, 2], bt[1, 0], bt[1, 31] = -1, kc.shape[0], 1 << 30
    out = paged_attention_forward(*[t.to(DEV) for t in (q, kc, vc, bt)], 16, sl.to(DEV)).cpu().double()
    assert float((out - _exact(q, kc, vc, bt, [100, 900])).abs().max()) <= 1e-5


def test_strided_caches_and_output():
    """K and V interleaved in one pool (different strides from a dense cache), and a transposed output."""
    q, kc, vc, bt, sl = _inputs([70, 1200], 8, 2, 128, 16, seed=4)
    both = torch.stack([kc, vc], dim=3).to(DEV)  # (pages, hkv, page, 2, d)
    out = torch.empty(8, 2, 128, device=DEV).transpose(0, 1)
    paged_attention_forward(q.to(DEV), both[:, :, :, 0], both[:, :, :, 1], bt.to(DEV), 16, sl.to(DEV), out=out)
    assert float((out.cpu().double() - _exact(q, kc, vc, bt, [70, 1200])).abs().max()) <= 1e-5
