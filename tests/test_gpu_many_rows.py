"""GPU: the row kernels over more rows than one launch holds (2^32 work-items: 2^26 rows at a
wave each), which go in slabs. A few rows hold values, at the ends and about the slabs' borders;
they must come out as from a call on those rows alone, and every other row as a row of zeros."""
import pytest
import torch

import vdn_fp8
from vdn_fp8.softmax_attention import qk_prep

pytestmark = pytest.mark.gpu

M = (1 << 26) + 5
ROWS = (0, 1, (1 << 23) - 1, 1 << 23, (1 << 24) + 1, (1 << 26) - 1, 1 << 26, M - 1)


def _rows(device, width, dtype):
    x = torch.zeros(M, width, device=device, dtype=dtype)
    at = torch.tensor(ROWS, device=device)
    some = torch.randn(len(ROWS), width, device=device, generator=torch.Generator(device=device).manual_seed(5)).to(dtype)
    x[at] = some
    return x, at, some


@pytest.mark.parametrize("name,width,dtype", [
    (n, w, d) for n, w in (("quantize_rows", 8), ("swiglu_quantize", 16), ("requantize_weight", 8), ("gelu_quantize", 8))
    for d in (torch.bfloat16, torch.float16) if n != "gelu_quantize" or d == torch.bfloat16])
def test_quantizers(device, name, width, dtype):
    fn = getattr(vdn_fp8, name)
    print(f"{name} [{M}, {width}] {dtype}", flush=True)
    x, at, some = _rows(device, width, dtype)
    q, s = fn(x)[:2]
    want_q, want_s = fn(some)[:2]
    q, s = q.view(torch.uint8), s.reshape(-1)
    assert torch.equal(q[at], want_q.view(torch.uint8)) and torch.equal(s[at], want_s.reshape(-1))
    zero_q, zero_s = fn(torch.zeros(1, width, device=device, dtype=dtype))[:2]
    assert int((s != zero_s.reshape(-1)).sum()) == len(ROWS)
    assert int((q.view(torch.int64) != zero_q.view(torch.uint8).view(torch.int64)).sum()) == len(ROWS)


def test_gated_residual_and_qk_prep(device):
    print(f"gated residual [{M}, 8], qk prep [{M}, 1, 64]", flush=True)
    x, at, some = _rows(device, 8, torch.bfloat16)
    gate = torch.ones(1, 8, device=device, dtype=torch.bfloat16)
    out = vdn_fp8.fused_block.post(x, gate, torch.zeros(M, device=device, dtype=torch.int32), x)
    assert torch.equal(out[at], some + some)
    out[at] = 0
    assert not bool(out.view(torch.int64).any())
    del x, out
    x, at, some = _rows(device, 64, torch.bfloat16)
    out = qk_prep(x.view(M, 1, 64), None, 1e-6)
    assert torch.equal(out[at].reshape(-1, 64), qk_prep(some.view(-1, 1, 64), None, 1e-6).reshape(-1, 64))
    out[at] = 0
    assert not bool(out.view(torch.int64).any())
