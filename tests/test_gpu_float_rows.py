"""GPU: float16 / float32 rows through the one-read quantizers and the GEMM's typed output.

The quantizer's row widths cover each register count's edges and the two-sweep kernel below
and past them; besides ordinary values every row holds elements at, one ulp below and one above each
e4m3 rounding boundary times the row's scale, where a quotient off by one ulp would change
the code. The GEMM's float16 / float32 output with its bias must give the bits of the binary32
product followed by torch's own cast and add."""
import numpy as np
import pytest
import torch

import oracle as O
import vdn_fp8
import vdn_fp8._lib as L
from conftest import codes, same_codes

pytestmark = pytest.mark.gpu


def _boundaries():
    """The positive midpoints between neighbouring e4m3 values (and zero), in float64."""
    c = torch.arange(0, 127, dtype=torch.uint8).view(torch.float8_e4m3fn).double().numpy()
    return (c[1:] + c[:-1]) / 2


def _row(rng, K, dtype, amax):
    t = np.float32 if dtype == torch.float32 else np.float16
    x = rng.standard_normal(K) * amax / 6
    scale = np.float64(np.float32(np.float32(t(amax)) / np.float32(448.0)))
    b = t(_boundaries() * scale)
    near = np.concatenate([b, np.nextafter(b, t(np.inf)), np.nextafter(b, t(0))])[:max(0, K - 1)]
    x = t(np.clip(x, -amax, amax))
    at = rng.permutation(K - 1)[:near.size] + 1
    x[at] = near * t(rng.choice([-1, 1]))
    x[0] = t(amax)
    return np.clip(x, -t(amax), t(amax))


@pytest.mark.parametrize("weight", [False, True])
@pytest.mark.parametrize("dtype,widths", [
    (torch.float32, (8, 768, 776, 1016, 1024, 1032, 4096, 5120, 8192, 12296, 16384, 16392)),
    (torch.float16, (8, 1024, 1032, 1536, 1544, 2040, 2048, 2056, 8192, 13824, 24576, 32768, 32776))])
def test_float_rows_bit_exact(device, dtype, widths, weight):
    rng = np.random.default_rng(5)
    for K in widths:
        print(f"float rows {dtype} K={K} weight={weight}", flush=True)
        rows = [_row(rng, K, dtype, a) for a in (1.0, 3.7, 448.0, 1.5e-3, 6.1e4 if dtype == torch.float16 else 3e38)]
        x = torch.from_numpy(np.stack(rows + [np.zeros_like(rows[0]), -rows[0]]))
        if weight:
            q, s = vdn_fp8.requantize_weight(x.to(device))
            want_q, want_s = O.quantize_weight_float(x.numpy())
        else:
            q, s = vdn_fp8.quantize_rows(x.to(device))
            want_q, want_s = O.quantize_rows_float(x.numpy())
        assert same_codes(codes(q), want_q).all()
        assert np.array_equal(s.cpu().numpy().reshape(-1).view(np.uint32), want_s.view(np.uint32))


def test_more_rows_than_workgroups_in_a_launch(device):
    """2^24 rows and more, which a launch of one 256-thread workgroup per row cannot hold."""
    M, K = (1 << 24) + 5, 8
    print(f"float rows [{M}, {K}]", flush=True)
    x = torch.zeros(M, K, device=device, dtype=torch.float16)
    rows = torch.tensor([0, 1, 255, 1 << 16, (1 << 24) - 1, 1 << 24, M - 1], device=device)
    x[rows] = torch.randn(rows.numel(), K, device=device, generator=torch.Generator(device=device).manual_seed(3)).half()
    q, s = vdn_fp8.quantize_rows(x)
    want_q, want_s = O.quantize_rows_float(x[rows].cpu().numpy())
    assert same_codes(codes(q[rows]), want_q).all()
    assert np.array_equal(s[rows].cpu().numpy().reshape(-1).view(np.uint32), want_s.view(np.uint32))
    assert int((s != s[2 ** 20 + 1]).sum()) == rows.numel() and int((q.view(torch.uint8).sum(1) != 0).sum()) == rows.numel()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 4, 16), (77, 260, 400), (700, 1032, 2048), (4096, 4096, 512), (520, 1028, 8192)])
def test_typed_output_is_the_cast_and_the_add(device, dtype, M, N, K):
    """(4096, 4096: whole rounds of the persistent kernel; 520 x 1028 x 8192: split along K.)"""
    print(f"typed gemm {dtype} [{M}, {N}, {K}]", flush=True)
    g = torch.Generator(device=device).manual_seed(M + N + K)
    lin = torch.nn.Linear(K, N, device=device, dtype=dtype)
    with torch.no_grad():
        lin.weight.copy_(0.02 * torch.randn(N, K, device=device, generator=g))
        lin.bias.copy_(torch.randn(N, device=device, generator=g))
    f = vdn_fp8.Fp8Linear(lin)
    xq, xs = vdn_fp8.quantize_rows((3 * torch.randn(M, K, device=device, generator=g)).to(dtype))
    xs[0] *= 1e9                       # float16 outputs that overflow
    with torch.no_grad():
        got = f.forward_quantized(xq, xs, out_dtype=dtype)
    ws = torch.empty(max(16, vdn_fp8.fp8_linear.gemm_workspace_bytes(M, N, K, xq.device)), device=device, dtype=torch.uint8)
    prod = torch.empty(M, N, device=device, dtype=torch.float32)
    ptr = lambda t: t.data_ptr()
    L.check(L.load().vdn_fp8_gemm_ws(ptr(xq), ptr(xs), ptr(f.weight_fp8), ptr(f.weight_scale), M, N, K, K, K, None,
                                     L.EPI_F32, None, None, 0, 0, None, 0, ptr(prod), N, ptr(ws), ws.numel(),
                                     torch.cuda.current_stream().cuda_stream), "gemm")
    want = prod.to(dtype) + f.bias.detach()
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # a bias that takes a gradient, or of another type, keeps the reference's own op
    assert f.forward_quantized(xq, xs, out_dtype=dtype).requires_grad
    f.bias = torch.nn.Parameter(f.bias.detach().double(), requires_grad=False)
    assert f.forward_quantized(xq, xs, out_dtype=dtype).dtype == torch.float64


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 132, 1040), (65, 1028, 1136), (0, 64, 2064), (333, 260, 4112), (300, 512, 8208)])
def test_forward_on_whole_lines(device, M, N, K, dtype):
    """`Fp8Linear.forward` spaces the codes of such widths by whole 128-byte lines: the output is
    bit for bit that of contiguous codes, also where every byte past a row's K is a NaN code."""
    g = torch.Generator(device=device).manual_seed(K + M)
    lin = torch.nn.Linear(K, N, dtype=dtype, device=device)
    f = vdn_fp8.Fp8Linear(lin)
    x = torch.randn(2, M, K, device=device, generator=g).to(dtype)   # (three dimensions: also without rows)
    with torch.no_grad():
        if M == 0:
            with pytest.raises(RuntimeError):
                f(x[0])          # as torch's reshape to (0, -1) refuses it
            return
        q, s = vdn_fp8.quantize_activation(x.reshape(-1, K))
        want = f.forward_quantized(q, s, out_dtype=dtype)
        padded = torch.full((2 * M, -(-K // 128) * 128), 0x7F, device=device, dtype=torch.uint8)
        padded[:, :K] = q.view(torch.uint8)
        got = f.forward_quantized(padded.view(torch.float8_e4m3fn)[:, :K], s, out_dtype=dtype)
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(got.view(bits), want.view(bits))
        assert torch.equal(f(x).reshape(-1, N).view(bits), want.view(bits))
