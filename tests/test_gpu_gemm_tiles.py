"""GPU: the GEMM's tile shapes against one another, bit for bit.

Every output is one chain of MFMAs over the 128-byte K blocks in ascending order followed by
the same roundings, so it may not depend on the tile it falls in, on the K rows' padding
with zero codes, or on the epilogue's store path. The problem is run as it is (by the
plan that its row names: the tile kernel, 224-row tiles, a last round in parts, or whole tiles
through the general epilogue) and inside one of exactly two rounds of whole 256 x 256 tiles of
the persistent kernel through the fast epilogue (the only one of a typed output is the general
one), its rows, columns and K padded."""
import pytest
import torch

import vdn_fp8
import vdn_fp8._lib as L
from conftest import gemm_plan

pytestmark = pytest.mark.gpu

MB, NB = 4096, 8192          # 16 x 32 tiles: two rounds on 256 compute units
_TYPED = {"f16": (torch.float16, L.DTYPE_F16), "f32": (torch.float32, L.DTYPE_F32)}


def _gemm(xq, sx, wq, sw, bias, epi, gate, gi, res, n):
    """vdn_fp8_gemm, or with epi "f16" / "f32" vdn_fp8_gemm_typed of that output and bias."""
    M, K = xq.shape
    ptr = lambda t: None if t is None else t.data_ptr()
    a, st = (ptr(xq), ptr(sx), ptr(wq), ptr(sw), M, n, K, K, K, ptr(bias)), torch.cuda.current_stream().cuda_stream
    if epi in _TYPED:
        dtype, code = _TYPED[epi]
        out = torch.empty(M, n, device=xq.device, dtype=dtype)
        L.check(L.load().vdn_fp8_gemm_typed(*a, code, ptr(out), n, None, 0, st), "gemm")
        return out
    out = torch.empty(M, n, device=xq.device, dtype=torch.bfloat16)
    L.check(L.load().vdn_fp8_gemm(*a, epi, ptr(gate), ptr(gi), 0 if gate is None else gate.shape[0],
                                  0 if gate is None else n, ptr(res), 0 if res is None else n, ptr(out), n, st), "gemm")
    return out


def _pad(t, *shape):
    out = torch.zeros(*shape, device=t.device, dtype=t.dtype)
    out[tuple(slice(0, s) for s in t.shape)] = t
    return out


# plan: rows of the persistent kernel's tiles, tiles it runs whole, channels and tokens of the
# tile kernel's (on 256 compute units)
@pytest.mark.parametrize("M,N,K,epi,plan", [
    (1, 260, 16, "none", (0, 0, 128, 64)),             # the smallest: one token, one partial K block
    (65, 1032, 400, "gelu", (0, 0, 128, 64)),          # K past the last whole block
    (333, 516, 2048, "rows", (0, 0, 128, 64)),         # rows that are not 16-byte multiples: 8-byte pieces
    (2514, 516, 256, "bias", (0, 0, 128, 64)),
    (486, 4100, 272, "f32", (0, 0, 128, 96)),
    (643, 4104, 256, "gelu", (0, 0, 128, 96)),
    (2938, 800, 656, "rows", (0, 0, 128, 96)),
    (866, 4104, 1040, "rows", (0, 0, 128, 128)),       # table rows and residual
    (1481, 2580, 656, "f16", (0, 0, 128, 128)),        # a binary16 output with its bias
    (962, 4096, 256, "gate", (256, 0, 128, 128)),      # 64 tiles as quarters, one gate row
    (1026, 5376, 256, "rows", (0, 0, 128, 192)),
    (1026, 5376, 656, "bias", (0, 0, 128, 192)),
    (2021, 2124, 1296, "gate", (0, 0, 128, 192)),
    (649, 6400, 768, "rows", (0, 0, 192, 96)),
    (3431, 2476, 400, "gelu", (0, 0, 192, 96)),
    (3078, 1856, 656, "f16", (0, 0, 192, 128)),        # 16-byte binary16 rows
    (1772, 2524, 768, "rows", (0, 0, 192, 128)),
    (2951, 5376, 400, "rows", (0, 0, 256, 128)),
    (3437, 4580, 400, "f32", (0, 0, 256, 128)),
    (2317, 5376, 256, "gelu", (224, 231, 0, 0)),       # 224-row tiles of the persistent kernel
    (2317, 5376, 512, "rows", (224, 231, 0, 0)),
    (1928, 4096, 512, "bias", (256, 0, 256, 128)),     # 128 tiles as halves
    (2576, 7552, 2048, "rows", (256, 256, 256, 128)),  # a round, then halves
    (3697, 6012, 768, "f16", (256, 256, 256, 128)),
    (3392, 5192, 768, "gelu", (256, 256, 128, 128)),   # a round, then quarters
    (2619, 6724, 256, "f32", (256, 256, 128, 128)),
    (4000, 4704, 2048, "rows", (256, 256, 128, 128)),
    (4000, 4168, 2048, "rows", (256, 256, 128, 64)),   # a round, then eighths: rows and columns past the end
    (2128, 7456, 256, "gate", (256, 256, 128, 64)),
    (2836, 5644, 256, "f16", (256, 256, 128, 64)),
    (4000, 7420, 512, "none", (256, 464, 0, 0)),       # whole tiles through the general epilogue, in more
    (4000, 7420, 512, "gelu", (256, 464, 0, 0)),       # than one round
    (4000, 7420, 512, "gate", (256, 464, 0, 0)),
    (4000, 7420, 512, "rows", (256, 464, 0, 0)),
    (4000, 7420, 512, "f16", (256, 464, 0, 0)),
    (4000, 7424, 512, "f32", (256, 464, 0, 0)),
])
def test_tile_shapes_give_the_same_bits(device, M, N, K, epi, plan):
    print(f"gemm tiles [{M}, {N}, {K}] {epi}", flush=True)
    KB = -(-K // 256) * 256
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        p = gemm_plan(M, N, K, N % 8 == 0 and epi not in _TYPED, cus=0)
        assert p[:2] + p[4:] == plan and p[2:4] == (0, 0)
        assert gemm_plan(MB, NB, KB, epi not in _TYPED, cus=0) == (256, 512, 0, 0, 0, 0)
    g = torch.Generator(device=device).manual_seed(M + N + K)
    rand = lambda *s: torch.randn(*s, device=device, generator=g)
    xq, sx = vdn_fp8.quantize_rows(_pad(rand(M, K).to(torch.bfloat16), M, K))
    wq, sw = vdn_fp8.requantize_weight((0.02 * rand(N, K)).to(torch.bfloat16))
    sx = sx.reshape(-1)
    bias = None if epi == "none" else (0.1 * rand(N)).to(_TYPED[epi][0] if epi in _TYPED else torch.bfloat16)
    gate = gi = res = None
    code = epi if epi in _TYPED else {"none": L.EPI_NONE, "bias": L.EPI_NONE, "gelu": L.EPI_GELU_TANH}.get(epi, L.EPI_GATE)
    if epi == "gate":
        gate = rand(1, N).to(torch.bfloat16)
    if epi == "rows":
        gate, res = rand(3, N).to(torch.bfloat16), rand(M, N).to(torch.bfloat16)
        gi = torch.randint(-1, 4, (M,), device=device, generator=g, dtype=torch.int32)   # clamped into the table
    got = _gemm(xq, sx, wq, sw, bias, code, gate, gi, res, N)
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
