"""The float32 varlen prefill kernel (f32 matrix instructions) against 64-bit
softmax attention: tile and key-block edges (a tile is 32 (query, head) rows,
a key block 16 keys, dealt to four waves), GQA groups that do and do not
divide 32, q_len != k_len, more than 64 sequences (the other item order), a
sequence without keys, and non-finite V rows that no query may see through
the causal mask. Tolerance: an output is a mean of the V rows, whose 32-bit
rounding and sums of at most a few hundred terms stay within 1e-5 of values of
order 1 (about 1e-6 is measured)."""

import pytest
import torch

from tinyserver_amd.kernels import flash_attn_varlen_func

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _cu(lens):
    return torch.tensor([0] + lens).cumsum(0).to(torch.int32)


def _inputs(lq, lk, hq, hkv, d, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(sum(lq), hq, d, generator=g), torch.randn(sum(lk), hkv, d, generator=g),
            torch.randn(sum(lk), hkv, d, generator=g))


def _exact(q, k, v, lq, lk, causal):
    out = torch.empty(q.shape, dtype=torch.float64)
    group, qs, ks = q.shape[1] // k.shape[1], 0, 0
    for nq, nk in zip(lq, lk):
        for h in range(q.shape[1]):
            s = q[qs:qs + nq, h].double() @ k[ks:ks + nk, h // group].double().T * q.shape[2] ** -0.5
            seen = torch.ones(nq, nk, dtype=torch.bool)
            if causal:
                seen = torch.arange(nk)[None] <= torch.arange(nq)[:, None]
            p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
            vv = v[ks:ks + nk, h // group].double()
            for r in range(nq):  # only the rows a query sees (a non-finite unseen row does not count)
                out[qs + r, h] = p[r, seen[r]] @ vv[seen[r]]
        qs, ks = qs + nq, ks + nk
    return out


def _check(lq, lk, hq, hkv, d, causal, seed, poison=None):
    q, k, v = _inputs(lq, lk, hq, hkv, d, seed)
    if poison is not None:
        v[poison[0], :, ::3] = poison[1]
    cq, ck = _cu(lq).to(DEV), _cu(lk).to(DEV)
    out = flash_attn_varlen_func(q.to(DEV), k.to(DEV), v.to(DEV), cq, ck, max(lq), max(lk), causal).cpu().double()
    ref = _exact(q, k, v, lq, lk, causal)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(out[~fin & ~torch.isnan(ref)], ref[~fin & ~torch.isnan(ref)])
    err = float((out[fin] - ref[fin]).abs().max())
    print(f"{lq} {hq}/{hkv} x {d} causal={causal}: max_abs={err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv,d", [(4, 2, 128), (2, 2, 64), (6, 2, 128), (8, 1, 64), (40, 1, 128)])
def test_tile_edges(hq, hkv, d, causal):
    lens = [1, 15, 16, 17, 32, 33, 127, 130]
    _check(lens, lens, hq, hkv, d, causal, seed=hq + d)


@pytest.mark.parametrize("causal", [True, False])
def test_q_len_differs_from_k_len(causal):
    _check([5, 40, 64, 3], [9, 33, 200, 1], 4, 2, 128, causal, seed=3)


def test_many_sequences():
    lens = [1 + (7 * i) % 40 for i in range(70)]
    _check(lens, lens, 4, 2, 128, True, seed=4)


def test_sequence_without_keys():
    lq, lk = [16, 40], [0, 50]
    q, k, v = _inputs(lq, lk, 4, 2, 128, 5)
    out = flash_attn_varlen_func(q.to(DEV), k.to(DEV), v.to(DEV), _cu(lq).to(DEV), _cu(lk).to(DEV), 40, 50,
                                 False).cpu().double()
    assert torch.isnan(out[:16]).all()
    assert float((out[16:] - _exact(q[16:], k, v, [40], [50], False)).abs().max()) <= 1e-5


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_unseen_non_finite_values(value):
    """A key's non-finite V row reaches the queries at or after it and no earlier one."""
    _check([20, 100], [20, 100], 4, 2, 128, True, seed=6, poison=(20 + 70, value))
