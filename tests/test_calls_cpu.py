"""The native host side of calls: loaded with the library, and everything but plain device tensors is left to Python."""
import pytest
import torch


def test_native_calls_leave_the_rest_to_python():
    from vllm_hymeta import _C
    _C.load()
    if _C.calls is None:
        pytest.skip("hymeta_calls.so is not built")
    q, starts = torch.zeros(2, 4, 128, dtype=torch.bfloat16), torch.zeros(3, dtype=torch.int32)
    state, decay = torch.zeros(2, 4, 128, 128), torch.ones(4)
    for args in ((), (q,), (None,) * 13, (q, q, q, state, starts, starts, starts, 1, decay, None, None, None, 0), ("q", 1, 2.0),
                 (q.numpy,) * 13, (torch.nn.Parameter(q.float()),) * 13):
        assert _C.calls.decay_scan(*args) is None
    for name in ("sink_attention", "meta_swa_paged_decode", "meta_swa_prefill", "lightning_attention", "delta_rule"):
        assert getattr(_C.calls, name)(*[q] * 26) is None and getattr(_C.calls, name)() is None
    with pytest.raises(TypeError):
        _C.calls.setup(_C)
