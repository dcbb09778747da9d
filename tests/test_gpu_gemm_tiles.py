"""GPU: the GEMM's tile shapes against one another, bit for bit.

Every output is one chain of MFMAs over the 128-byte K blocks in ascending order followed by
the same roundings, so it may not depend on the tile it falls in, on the K rows' padding
with zero codes, or on the epilogue's store path. The problem is run as it is (the plan
picks the tile kernel, 224-row tiles or a last round in parts) and inside one of exactly two
rounds of whole 256 x 256 tiles of the persistent kernel, its rows, columns and K padded."""
import pytest
import torch

import vdn_fp8
import vdn_fp8._lib as L
from conftest import gemm_plan

pytestmark = pytest.mark.gpu

MB, NB = 4096, 8192          # 16 x 32 tiles: two rounds on 256 compute units


def _gemm(xq, sx, wq, sw, bias, epi, gate, gi, res, n):
    M, K = xq.shape
    out = torch.empty(M, n, device=xq.device, dtype=torch.float32 if epi == L.EPI_F32 else torch.bfloat16)
    ptr = lambda t: None if t is None else t.data_ptr()
    L.check(L.load().vdn_fp8_gemm(ptr(xq), ptr(sx), ptr(wq), ptr(sw), M, n, K, K, K, ptr(bias), epi, ptr(gate), ptr(gi),
                                  0 if gate is None else gate.shape[0], 0 if gate is None else n, ptr(res),
                                  0 if res is None else n, ptr(out), n, torch.cuda.current_stream().cuda_stream), "gemm")
    return out


def _pad(t, *shape):
    out = torch.zeros(*shape, device=t.device, dtype=t.dtype)
    out[tuple(slice(0, s) for s in t.shape)] = t
    return out


@pytest.mark.parametrize("M,N,K,epi", [
    (1, 260, 16, "none"),             # the smallest: one token, one partial K block
    (65, 1032, 400, "gelu"),          # 128 x 64 tiles, K past the last whole block
    (333, 516, 2048, "rows"),         # rows that are not 16-byte multiples: 8-byte pieces
    (2514, 516, 256, "bias"),         # 128 x 96
    (486, 4100, 272, "f32"),          # 128 x 128
    (866, 4104, 1040, "rows"),        # 128 x 192, table rows and residual
    (643, 4104, 256, "gelu"),         # 192 x 96
    (962, 4096, 256, "gate"),         # 192 x 128, one gate row
    (1026, 5376, 256, "rows"),        # 256 x 128
    (1026, 5376, 656, "bias"),
    (2317, 5376, 256, "gelu"),        # 224-row tiles of the persistent kernel
    (2317, 5376, 512, "rows"),
    (1928, 4096, 512, "bias"),        # 128 tiles as halves
    (4000, 4168, 2048, "rows"),       # one round and a last one in eighths, columns past N
    (4000, 4704, 2048, "rows"),       # one round and a last one in quarters
])
def test_tile_shapes_give_the_same_bits(device, M, N, K, epi):
    print(f"gemm tiles [{M}, {N}, {K}] {epi}", flush=True)
    g = torch.Generator(device=device).manual_seed(M + N + K)
    rand = lambda *s: torch.randn(*s, device=device, generator=g)
    xq, sx = vdn_fp8.quantize_rows(_pad(rand(M, K).to(torch.bfloat16), M, K))
    wq, sw = vdn_fp8.requantize_weight((0.02 * rand(N, K)).to(torch.bfloat16))
    sx = sx.reshape(-1)
    bias = (0.1 * rand(N)).to(torch.bfloat16) if epi != "f32" else None
    gate = gi = res = None
    code = {"none": L.EPI_NONE, "bias": L.EPI_NONE, "gelu": L.EPI_GELU_TANH, "f32": L.EPI_F32}.get(epi, L.EPI_GATE)
    if epi == "none":
        bias = None
    if epi == "gate":
        gate = rand(1, N).to(torch.bfloat16)
    if epi == "rows":
        gate, res = rand(3, N).to(torch.bfloat16), rand(M, N).to(torch.bfloat16)
        gi = torch.randint(-1, 4, (M,), device=device, generator=g, dtype=torch.int32)   # clamped into the table
    got = _gemm(xq, sx, wq, sw, bias, code, gate, gi, res, N)
    KB = -(-K // 256) * 256
    u8 = lambda t, *s: _pad(t.view(torch.uint8), *s).view(torch.float8_e4m3fn)
    want = _gemm(u8(xq, MB, KB), _pad(sx, MB), u8(wq, NB, KB), _pad(sw, NB), None if bias is None else _pad(bias, NB),
                 code, None if gate is None else _pad(gate, gate.shape[0], NB), None if gi is None else _pad(gi, MB),
                 None if res is None else _pad(res, MB, NB), NB)[:M, :N]
    torch.cuda.synchronize()
    bits = torch.int32 if epi == "f32" else torch.int16
    assert torch.equal(got.view(bits), want.contiguous().view(bits))


@pytest.mark.parametrize("M,N,K,out", [(2817, 28672, 8192, "f16"), (3329, 28676, 8192, "bf16")])
def test_the_answered_workspace_is_enough(device, M, N, K, out):
    """A workspace of the queried size (at least 16 bytes, so that a pointer is given) serves rows
    that take the general epilogue too, where the query assumes 16-byte rows."""
    print(f"gemm workspace [{M}, {N}, {K}] {out}", flush=True)
    g = torch.Generator(device=device).manual_seed(M)
    code = lambda *s: torch.randint(0, 120, s, device=device, generator=g, dtype=torch.uint8).view(torch.float8_e4m3fn)
    xq, wq = code(M, K), code(N, K)
    sx, sw = (1e-4 * torch.rand(n, device=device, generator=g) for n in (M, N))
    ws = torch.empty(max(16, vdn_fp8.fp8_linear.gemm_workspace_bytes(M, N, K, device)), device=device, dtype=torch.uint8)
    st = torch.cuda.current_stream().cuda_stream
    lib, outs = L.load(), []
    for w, size in ((ws.data_ptr(), ws.numel()), (None, 0)):
        o = torch.empty(M, N, device=device, dtype=torch.float16 if out == "f16" else torch.bfloat16)
        a = (xq.data_ptr(), sx.data_ptr(), wq.data_ptr(), sw.data_ptr(), M, N, K, K, K)
        if out == "f16":
            L.check(lib.vdn_fp8_gemm_typed(*a, None, L.DTYPE_F16, o.data_ptr(), N, w, size, st), "gemm")
        else:
            L.check(lib.vdn_fp8_gemm_ws(*a, None, L.EPI_NONE, None, None, 0, 0, None, 0, o.data_ptr(), N, w, size, st), "gemm")
        outs.append(o)
    torch.cuda.synchronize()
    if ws.numel() == 16:
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))   # no split either way


def test_more_tiles_than_a_launch_holds(device):
    """2^24 workgroups of 256 threads pass what one launch starts: the rows go in halves."""
    M, N, K = 192 * (1 << 24) + 5, 4, 16
    need = M * (K + 4 + 2 * N)
    if torch.cuda.mem_get_info(device)[0] < need + (16 << 30):
        pytest.skip(f"needs {need >> 30} GiB of GPU memory")
    print(f"gemm [{M}, {N}, {K}], plan {gemm_plan(M, N, K, False, cus=0)}", flush=True)
    xq = torch.zeros(M, K, device=device, dtype=torch.uint8)
    rows = [0, 1, M // 2, M // 2 + 511, 192 * (1 << 24) - 1, 192 * (1 << 24), M - 1]
    for i, r in enumerate(rows):
        xq[r, i] = 0x38                                        # 1.0
    sx, sw = torch.ones(M, device=device), torch.arange(1.0, N + 1, device=device)
    wq = torch.full((N, K), 0x38, device=device, dtype=torch.uint8)
    out = torch.full((M, N), 7.0, device=device, dtype=torch.bfloat16)
    st = torch.cuda.current_stream().cuda_stream
    L.check(L.load().vdn_fp8_gemm(xq.data_ptr(), sx.data_ptr(), wq.data_ptr(), sw.data_ptr(), M, N, K, K, K, None, L.EPI_NONE,
                                  None, None, 0, 0, None, 0, out.data_ptr(), N, st), "gemm")
    torch.cuda.synchronize()
    for r in rows:
        assert torch.equal(out[r].float(), sw), r
        out[r] = 0
    assert not any(bool(out[i:i + (1 << 28)].any()) for i in range(0, M, 1 << 28))
    del xq, sx, out
    torch.cuda.empty_cache()
