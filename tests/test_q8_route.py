"""Which int8 matvec calls quantize their rows in a launch of their own (quant_q8) and which in the matvec kernel: the
K-sliced Q4_K kernel keeps its one launch wherever the int8 MFMA does not take the planar buffer (fewer than nine tokens,
or fewer than 32768 outputs)."""
import pytest

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("fmt,n,k,tokens,staged", [
    ("q4_k", 1024, 4096, 8, True), ("q4_k", 1024, 4096, 9, True), ("q4_k", 1024, 4096, 31, True),
    ("q4_k", 1024, 4096, 32, False), ("q4_k", 12288, 4096, 8, True), ("q4_k", 12288, 4096, 9, False),
    ("q4_k", 100, 8192, 300, True), ("q4_k", 4096, 2048, 1, False),
    ("q4_kt", 1024, 4096, 2, True), ("q4_kt", 1024, 4096, 3, False), ("q6_k", 1024, 4096, 1, False)])
def test_q8_input_route(monkeypatch, fmt, n, k, tokens, staged):
    import qmm.ops as ops
    calls = []
    monkeypatch.setattr(ops, "quant_q8", lambda x: calls.append(x.shape) or torch.empty(0, dtype=torch.uint8))
    x = torch.zeros((tokens, k), dtype=torch.bfloat16)
    got, code, count = ops._q8_input(fmt, x, n, k, None, staged_tokens=2)
    assert count == tokens
    assert (got is x, not calls, code == ops.DTYPE["bf16"]) == (staged, staged, staged)
