"""The _tsa_host extension describes tensors as the ctypes route does: the
same argument errors from the C entry points (which check everything before any
device work) for the same tensors, None as a NULL view, the entry points'
argument counts, and the general route for tensor subclasses."""

import pytest
import torch

from tinyserver_amd import _lib


def _decode_args(dtype=torch.bfloat16, heads=8, strided=False):
    q = torch.zeros(3, heads, 128, dtype=dtype)
    kc = torch.zeros(4, 2, 16, 256, dtype=dtype)[..., ::2] if strided else torch.zeros(4, 2, 16, 128, dtype=dtype)
    return [q, q, kc, kc, torch.zeros(3, 2, dtype=torch.int32), torch.zeros(3, dtype=torch.int32)]


def _both(name, *args):
    got = _lib.call(name, *args), _lib.load().tsa_last_error()
    want = getattr(_lib.load(), name)(*(a if isinstance(a, (int, float)) else _lib.view(a) for a in args))
    assert got == (want, _lib.load().tsa_last_error())
    return got


def test_same_status_and_message():
    for args in (_decode_args(heads=7), _decode_args(torch.float16, heads=3)):  # not a multiple of 2 kv heads
        rc, msg = _both("tsa_paged_decode", *args, 0.1, 0, 0, 0, 0)
        assert rc == _lib.TSA_ERR_INVALID and b"multiple" in msg
    a = _decode_args()
    rc, msg = _both("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)  # (strides, sizes and dtypes passed: no workspace)
    assert rc == _lib.TSA_ERR_INVALID and b"workspace of 0 bytes is too small" in msg
    a[4] = a[4].long()
    assert b"int32" in _both("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)[1]
    a = _decode_args()
    a[3] = None
    assert b"4D" in _both("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)[1]
    a[3] = torch.zeros(4, 2, 16, 64, dtype=torch.bfloat16)
    assert b"match" in _both("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)[1]


def test_what_has_no_view_is_refused():
    a = _decode_args()
    a[0] = torch.zeros(1, 1, 1, 1, 1)
    with pytest.raises(ValueError, match="rank > 4"):
        _lib.call("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)
    a[0] = torch.zeros(3, 8, 128, dtype=torch.float64)
    with pytest.raises(ValueError, match="unsupported dtype"):
        _lib.call("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0)
    with pytest.raises(TypeError, match="tsa_paged_decode takes 6 tensors"):
        _lib.call("tsa_paged_decode", *_decode_args(), 0.1, 0, 0, 0)
    with pytest.raises(TypeError):
        _lib.call("tsa_paged_decode", *([None] * 40))
    with pytest.raises(RuntimeError):  # no storage to point at: a Python error, no abort
        a[0] = torch.zeros(3, 8, 128, dtype=torch.bfloat16, device="meta")
        torch.func.vmap(lambda x: _lib.call("tsa_paged_decode", x, *_decode_args()[1:], 0.1, 0, 0, 0, 0) or x)(
            torch.zeros(2, 3, 8, 128, dtype=torch.bfloat16))


def test_tensor_subclasses_take_the_general_route():
    class Sub(torch.Tensor):
        pass

    a = _decode_args(heads=7)
    a[1] = a[1].as_subclass(Sub)
    assert _lib.host().call(0, *a, 0.1, 0, 0, 0, 0) is None
    assert _lib.call("tsa_paged_decode", *a, 0.1, 0, 0, 0, 0) == _lib.TSA_ERR_INVALID
    with pytest.raises(RuntimeError, match="GPU"):
        _lib.require_device(*a)


def test_entries_match_the_binding():
    names = _lib.host().entries()
    assert set(names) <= set(_lib.SIGNATURES)
    for name in names:
        kinds = _lib.SIGNATURES[name][1]
        assert len(kinds) == {"tsa_paged_decode": 11, "tsa_paged_decode_step": 18, "tsa_qk_norm_rope": 10,
                              "tsa_qk_norm_rope_store": 16, "tsa_varlen_prefill": 11, "tsa_mixed_attention": 19,
                              "tsa_sample_tokens": 7, "tsa_sample_tokens_ws": 9}[name]
