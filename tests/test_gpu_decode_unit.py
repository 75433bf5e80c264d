"""The unit form of the 16-bit paged decode (small block tables: one workgroup
a unit up to 512 tokens, splits of 256 tokens above) against 64-bit softmax
attention: tile, wave and split edges, GQA groups of 1 to 16, head_dim 64 and
128, pages of 4 to 256 tokens, strided cache rows, an empty sequence, page ids
outside the pool, non-finite slots past a sequence's end, tables on both sides
of the plan's limits; the fused step with its new token at those edges (and past
them, in the stream) and the one-launch prefill + decode, both bit-identical to
the calls they stand for.
Tolerance: the output is rounded to its type (bf16: 2^-9 of the value, f16:
2^-12), P keeps 16 (22) bits, so 2^-8 (2^-11) of values of order 1."""

import pytest
import torch

from tests.helpers import assert_bitexact
from tests.test_gpu_decode_f32 import _exact, _inputs
from tinyserver_amd.kernels import (mixed_attention, paged_attention_forward,
                                    paged_decode_step, qk_norm_rope_store)

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F16 = torch.bfloat16, torch.float16


def _cast(x, dtype):
    return tuple(t.to(dtype) if t.is_floating_point() else t for t in x)


@pytest.mark.parametrize("hq,hkv,d,page,dtype,lens", [
    (16, 8, 128, 16, BF, [0, 1, 15, 16, 17, 128, 129, 512]),        # 64 units, one workgroup each
    (32, 8, 128, 16, F16, [511, 385, 257, 3] * 4),                  # 128 units
    (16, 1, 128, 32, BF, [512, 100, 33]),
    (8, 8, 64, 16, BF, [496, 512, 1]),
    (6, 2, 128, 8, BF, [7, 8, 500, 9]),                             # pages of less than a tile
    (6, 2, 64, 4, F16, [509, 3, 64]),
    (16, 8, 128, 16, BF, [0, 1, 256, 257, 513, 528]),               # split units
    (32, 4, 128, 256, BF, [255, 256, 257, 4000, 1]),
    (6, 2, 128, 8, BF, [700, 8, 257]),
    (4, 4, 64, 16, F16, [3000, 1, 512]),
    (8, 2, 128, 16, BF, [9000, 300, 0]),                            # 36 splits: streaming loads
])
def test_against_64_bits(hq, hkv, d, page, dtype, lens):
    q, kc, vc, bt, sl = _cast(_inputs(lens, hq, hkv, d, page, seed=d + page + len(lens)), dtype)
    ref = _exact(q, kc, vc, bt, lens)
    for s, n in enumerate(lens):
        if n % page:
            kc[bt[s, n // page], :, n % page:] = float("nan")
            vc[bt[s, n // page], :, n % page:] = float("inf")
    out = paged_attention_forward(*[t.to(DEV) for t in (q, kc, vc, bt)], page, sl.to(DEV)).cpu().double()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    err = float((out - ref).nan_to_num().abs().max())
    print(f"{hq}/{hkv} x {d}, page {page}, {dtype}: max_abs={err:.2e}", flush=True)
    assert err <= (2 ** -8 if dtype == BF else 2 ** -11) * max(1.0, float(ref.nan_to_num().abs().max()))


@pytest.mark.parametrize("lens", [[100, 300], [100, 900]])
def test_page_ids_outside_the_pool_and_strided_rows(lens):
    q, kc, vc, bt, sl = _cast(_inputs(lens, 4, 2, 128, 16, seed=3), BF)
    bt[0, 2], bt[1, 0], bt[1, 17] = -1, kc.shape[0], 1 << 30
    ref = _exact(q, kc, vc, bt, lens)
    both = torch.stack([kc, vc], dim=3).to(DEV)
    for k, v in ((kc.to(DEV), vc.to(DEV)), (both[:, :, :, 0], both[:, :, :, 1])):
        out = paged_attention_forward(q.to(DEV), k, v, bt.to(DEV), 16, sl.to(DEV)).cpu().double()
        assert float((out - ref).abs().max()) <= 2 ** -8 * float(ref.abs().max())


@pytest.mark.parametrize("hq,hkv,page,dtype,lens", [
    (16, 8, 16, BF, [1, 16, 17, 129, 512]),
    (64, 8, 32, BF, [1, 500, 33]),                 # G = 8: the k row is a third wave's
    (2, 2, 16, F16, [256, 257, 1, 512, 513, 700]),
    (8, 2, 256, BF, [1, 255, 257, 3000, 4096]),
    (8, 4, 16, BF, [8193, 64]),
    # Past the unit form's limits (the stream), several tiles a wave: runs of
    # one-tile units, more of them in flight than a wave has unit buffers.
    (16, 8, 16, BF, [3000, 1, 17] * 7),
    (8, 8, 32, F16, [3000] * 6 + [16] * 6 + [33, 1] * 6),
    (2, 1, 16, BF, [33, 1, 17] * 501),             # the most sequences it takes
])
def test_fused_step_is_the_two_launches(hq, hkv, page, dtype, lens):
    g = torch.Generator().manual_seed(hq + page)
    b, d = len(lens), 128
    q, kc, vc, bt, sl = [t.to(DEV) for t in _cast(_inputs(lens, hq, hkv, d, page, seed=7), dtype)]
    if b > 2:
        bt[2, (lens[2] - 1) // page] = -1  # a new token without a page: not stored, not attended to
    k, v = (torch.randn(b, hkv, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    qw, kw = ((1 + 0.1 * torch.randn(d, generator=g)).to(dtype).to(DEV) for _ in range(2))
    ang = (sl.cpu() - 1)[:, None].float() / (1e6 ** (torch.arange(0, d, 2) / d))
    cos, sin = (torch.cat([f, f], -1).to(dtype).to(DEV) for f in (ang.cos(), ang.sin()))
    kc_a, vc_a, kc_b, vc_b = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    cu = torch.arange(b + 1, dtype=torch.int32, device=DEV)
    qa, _ = qk_norm_rope_store(q, k, v, qw, kw, cos, sin, 1e-6, kc_a, vc_a, bt, cu, sl - 1, return_k=False)
    out_a = paged_attention_forward(qa, kc_a, vc_a, bt, page, sl)
    out_b = paged_decode_step(q, k, v, qw, kw, cos, sin, 1e-6, kc_b, vc_b, bt, sl)
    torch.cuda.synchronize()
    assert_bitexact(vc_b, vc_a, "v cache")
    assert_bitexact(kc_b, kc_a, "k cache")
    assert_bitexact(out_b, out_a, f"fused step {lens}")


@pytest.mark.parametrize("lens", [[5, 300, 512, 17], [900, 257, 1]])
def test_mixed_decode_role(lens):
    """Four waves take the unit's virtual waves in turn: the same bits."""
    g = torch.Generator().manual_seed(9)
    q, kc, vc, bt, sl = [t.to(DEV) for t in _cast(_inputs(lens, 8, 2, 128, 16, seed=8), BF)]
    pq, pk, pv = (torch.randn(70, h, 128, generator=g).to(BF).to(DEV) for h in (8, 2, 2))
    cu = torch.tensor([0, 30, 70], dtype=torch.int32, device=DEV)
    _, out = mixed_attention(pq, pk, pv, cu, 40, q, kc, vc, bt, sl, prefill_workgroups=64)
    assert_bitexact(out, paged_attention_forward(q, kc, vc, bt, 16, sl), f"mixed decode {lens}")
