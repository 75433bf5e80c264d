"""The key-count pass of the sampler (bf16 rows of 16,384 to 155,648 logits; f16
rows, which never take it, beside them) against the histogram paths
(TSA_SAMPLE_CANDIDATES=0 in the environment): both add up the same integer masses
and compare them with the same targets, so the tokens are equal, over the row's forms (vocabulary sizes at the ends of the
range and beside a whole number of spans, heavy ties, both
zeros, -inf and lowest-value masks, one value only, NaN, +inf), temperatures,
top-k cuts of the candidate pass's (which sends rows of many ties on to the
key-count pass), above them and past the row's weight, top-p from 0
to past 1 and uniforms at both ends; and against the oracle in 64 bits."""

import pytest
import torch

from oracle import sampling as os_
from tinyserver_amd.kernels import sample_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(v, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(12, v, generator=g) * 2.5
    x[1] = (x[1] * 4).round() / 4                      # heavy ties
    x[2] = (x[2] > 0).float()                          # two values, tens of thousands of each
    x[3] = torch.where(x[3].abs() < 2, x[3].sign() * 0.0, x[3] - 20)  # both zeros
    x[4, torch.rand(v, generator=g) < 0.99] = float("-inf")
    x[5, torch.rand(v, generator=g) < 0.99] = torch.finfo(dtype).min
    x[6] = 1.5
    x[7] = -x[7].abs() - 3                             # negatives only
    x[8, v // 2] = 40
    x[9] = x[9] * 40
    x[10, 5] = float("nan")
    x[11, 7] = float("inf")
    return x.to(dtype).to(DEV)


PARAMS = [(1.0, 0, 0.95), (1.0, 0, 1.0), (0.7, 600, 0.9), (1.3, 10 ** 6, 0.5), (0.05, 0, 0.999), (30.0, 5000, 1.5),
          (1.0, 15000, 1.0), (1.0, 0, 0.0), (1e-5, 0, 0.9), (0.8, 50, 0.9), (1.0, 512, 1.0), (1.0, 1, 1.0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("v", [16384, 16392, 65536, 151936, 155648])
def test_same_tokens_as_the_histogram_paths(v, dtype, monkeypatch):
    x = _rows(v, dtype, seed=v)
    for i, (t, k, p) in enumerate(PARAMS):
        args = [torch.full((12,), val, dtype=dt, device=DEV) for val, dt in
                ((t, torch.float32), (k, torch.int64), (p, torch.float32))]
        for u in (0.0, 0.37, 0.999999):
            un = torch.full((12,), u, device=DEV)
            got = sample_tokens(x, *args, un).tolist()
            monkeypatch.setenv("TSA_SAMPLE_CANDIDATES", "0")
            want = sample_tokens(x, *args, un).tolist()
            monkeypatch.delenv("TSA_SAMPLE_CANDIDATES")
            assert got == want, (v, dtype, t, k, p, u)
    print(f"V {v} {dtype}: equal", flush=True)


def test_strided_rows_and_the_oracle(monkeypatch):
    """Rows of a wider buffer (a 16-byte aligned stride, then one that leaves every other row misaligned)."""
    g = torch.Generator().manual_seed(1)
    for width in (16392, 16388):
        x = (torch.randn(8, width, generator=g) * 3).to(torch.bfloat16)[:, :16384]
        un = torch.rand(8, generator=g)
        t, k, p = torch.full((8,), 0.9), torch.zeros(8, dtype=torch.int64), torch.full((8,), 0.8)
        wide = torch.empty(8, width, dtype=torch.bfloat16, device=DEV)
        wide[:, :16384] = x.to(DEV)
        got = sample_tokens(wide[:, :16384], t.to(DEV), k.to(DEV), p.to(DEV), un.to(DEV)).tolist()
        want = os_.sample_tokens(x, t, k, p, un, dtype=torch.float64).tolist()
        for r in range(8):
            if got[r] != want[r]:  # only where the decision lies within 32-bit rounding of its target
                assert os_.decision_margin(x[r], 0.9, 0, 0.8, float(un[r])) < 1e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_no_workspace_where_none_is_read(dtype):
    """bf16 rows the key-count pass takes, and float32 rows, bring none (f16: 32 MB here)."""
    x = torch.randn(64, 151936, device=DEV).to(dtype)
    args = [torch.full((64,), val, dtype=dt, device=DEV) for val, dt in
            ((1.0, torch.float32), (0, torch.int64), (0.95, torch.float32), (0.5, torch.float32))]
    sample_tokens(x, *args)
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    sample_tokens(x, *args)
    assert torch.cuda.max_memory_allocated() - before < 1 << 16


@pytest.mark.parametrize("b", [3, 64, 86])
def test_longer_rows_split(b):
    """bf16 rows past the key-count pass's range: the split launches (with and
    without bucket lists) against one workgroup a row (rows that start 2 bytes
    off a 16-byte boundary)."""
    g = torch.Generator().manual_seed(b)
    v = 163840
    x = (torch.randn(b, v, generator=g) * 2.5).to(torch.bfloat16).to(DEV)
    odd = torch.empty(b, v + 8, dtype=torch.bfloat16, device=DEV)[:, 1:v + 1]
    odd.copy_(x)
    args = [torch.full((b,), val, dtype=dt, device=DEV) for val, dt in
            ((1.0, torch.float32), (0, torch.int64), (0.95, torch.float32))] + [torch.rand(b, generator=g).to(DEV)]
    assert sample_tokens(x, *args).tolist() == sample_tokens(odd, *args).tolist()
