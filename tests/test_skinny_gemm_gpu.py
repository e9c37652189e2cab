"""cdssm_skinny_gemm (decode-size linear layers) against a float32 reference.

The reference is the unfused computation the decode step would otherwise run:
the model's RMSNorm (x * rsqrt(mean(x^2) + eps), rounded to bf16, times the
norm weight, rounded again), then the product in float32 from the bf16
operands, plus bias and residual.  The kernel rounds x * w_norm (not the
normalised x) to bf16 and applies the row scale to the float32 result, so the
two differ by bf16 rounding of the operands: tolerance 1e-2 normwise on the
bf16 output (max |y - ref| / max |ref|), 5e-3 without the norm (the output's
rounding to bf16, up to half a unit in the last place = 2^-8 relative, and the
summation order).
"""

import pytest
import torch

from _gpu_util import DEV, log, rel

pytestmark = pytest.mark.gpu


def _reference(x, w, bias=None, residual=None, norm_weight=None, eps=0.0):
    x32 = x.float()
    if norm_weight is not None:
        xn = (x32 * torch.rsqrt(x32.pow(2).mean(-1, keepdim=True) + eps)).to(torch.bfloat16)
        x32 = (xn * norm_weight.to(torch.bfloat16)).float()
    y = x32 @ w.float().t()
    if bias is not None:
        y = y + bias.float()
    if residual is not None:
        y = y + residual.float()
    return y


@pytest.mark.parametrize("name,M,K,N,use_bias,use_res,use_norm", [
    ("in_proj + RMSNorm", 64, 1024, 3104, True, False, True),
    ("gate/Q stacked", 64, 1024, 1136, True, False, False),
    ("out_proj + residual", 64, 1024, 1024, False, True, False),
    ("tied head + RMSNorm", 64, 1024, 32000, False, False, True),
    ("ragged rows and columns", 7, 256, 45, True, True, True),
    ("K 2048 (d_inner of the reference config)", 64, 2048, 1024, False, True, False),
    ("K 384: four waves", 33, 384, 100, True, False, True),
    ("one row", 1, 128, 16, False, False, False),
])
def test_skinny_gemm_matches_fp32_reference(name, M, K, N, use_bias, use_res, use_norm):
    from cdssm_hip.lm import skinny_linear
    g = torch.Generator().manual_seed(M * 7 + N)
    x = (torch.randn(M, K, generator=g) * 2.0).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    bias = (torch.randn(N, generator=g) * 0.1).to(torch.bfloat16) if use_bias else None
    res = torch.randn(M, N, generator=g).to(torch.bfloat16) if use_res else None
    nw = (1.0 + 0.1 * torch.randn(K, generator=g)).to(torch.bfloat16) if use_norm else None
    eps = 1e-5
    log(f"[skinny gemm] {name}: M{M} K{K} N{N}")
    y = skinny_linear(x.to(DEV), w.to(DEV), None if bias is None else bias.to(DEV),
                      None if res is None else res.to(DEV), None if nw is None else nw.to(DEV), eps)
    torch.cuda.synchronize()
    ref = _reference(x, w, bias, res, nw, eps)
    e = rel(y.float().cpu(), ref)
    log(f"   rel err {e:.2e}")
    assert e <= (1e-2 if use_norm else 5e-3), (name, e)


def test_skinny_gemm_strided_rows_and_graph_replay():
    """x a column slice of a wider buffer (row stride > K); the call captured in a HIP
    graph and replayed on rewritten inputs gives the eager result each time."""
    from cdssm_hip.lm import skinny_linear
    M, K, N = 64, 1024, 1136
    g = torch.Generator().manual_seed(3)
    buf = torch.randn(M, K + 128, generator=g).to(torch.bfloat16).to(DEV)
    x = buf[:, 128:]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).to(DEV)
    b = torch.randn(N, generator=g).to(torch.bfloat16).to(DEV)
    y_eager = skinny_linear(x, w, b)
    torch.cuda.synchronize()
    assert rel(y_eager.float().cpu(), _reference(x.cpu(), w.cpu(), b.cpu())) <= 5e-3
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_g = skinny_linear(x, w, b)
    for seed in (4, 5, 4):
        buf.copy_(torch.randn(M, K + 128, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16))
        graph.replay()
        torch.cuda.synchronize()
        ref = skinny_linear(x, w, b)
        torch.cuda.synchronize()
        assert torch.equal(y_g.cpu(), ref.cpu()), seed
    log("[skinny gemm] strided rows, graph replays equal eager calls")


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("M,N", [
    (64, 1152), (64, 1153), (64, 2304), (64, 2305),  # 16 | 32 and 32 | 64 rows per workgroup, M = 64
    (48, 1536), (48, 1537), (33, 2304), (33, 2320),  # three row groups of 16, the last one of a single row
    (17, 2304), (17, 2305), (17, 4609),              # two groups of 16, then one of 32 (the third tile unused)
    (16, 4608), (1, 4609), (64, 7), (17, 127),       # one group; fewer column tiles than XCDs
])
def test_rows_per_workgroup_leave_the_sums_alone(M, N, norm):
    """16, 32 or 64 rows go to a workgroup by M and N.  The order of every sum is the same for all of them, so
    each row equals, bit for bit, the product of that row alone; that one is within the rounding of its bf16
    result (2^-8 relative to the largest output) and, with the norm, of its operand (2^-8 again) of a 64-bit
    product of the same operands."""
    from cdssm_hip.lm import skinny_linear
    K = 256
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(N, K, generator=g) / 16.0).to(torch.bfloat16).to(DEV)
    bias = torch.randn(N, generator=g).to(torch.bfloat16).to(DEV)
    res = torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV)
    nw = (1.0 + 0.1 * torch.randn(K, generator=g)).to(torch.bfloat16).to(DEV) if norm else None
    y = skinny_linear(x, w, bias, res, nw, 1e-5)
    for m in sorted({0, 15, 16, 31, 32, M - 1} & set(range(M))):
        one = skinny_linear(x[m:m + 1], w, bias, res[m:m + 1], nw, 1e-5)
        assert torch.equal(y[m:m + 1], one), f"row {m}"
    x64 = x.double()
    if norm:
        x64 = x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    ref = (x64 @ w.double().t() + bias.double() + res.double()).cpu()
    assert rel(y.double().cpu(), ref) <= (2 if norm else 1) * 2.0 ** -8 + 1e-5


@pytest.mark.parametrize("M,N,col,C,taps", [
    (64, 3104, 1024, 1024, 4),  # in_proj of the decode step; 64 rows per workgroup
    (33, 45, 7, 30, 8), (1, 16, 0, 16, 1), (17, 40, 24, 16, 2), (64, 2304, 1, 2303, 3),
])
def test_conv_step_in_the_product(M, N, col, C, taps):
    """The product and the conv step on its columns in one launch, over two tokens, against the two launches: the
    same arithmetic on the same rounded values, equal bits in the product, the conv's output and the window."""
    from cdssm_hip.lm import conv1d_silu_step, skinny_linear, skinny_linear_conv_step
    K, g = 256, torch.Generator().manual_seed(N + taps)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)

    w, b, nw, cw, cb, win = rnd(N, K), rnd(N), rnd(K), rnd(C, 1, taps), rnd(C), rnd(M, taps - 1, C)
    win2 = win.clone()
    for _ in range(2):
        x = rnd(M, K)
        y, yc = skinny_linear_conv_step(x, w, b, nw, 1e-5, col, win, cw, cb)
        want = skinny_linear(x, w, b, norm_weight=nw, eps=1e-5)
        assert torch.equal(y, want)
        assert torch.equal(yc, conv1d_silu_step(want[:, col:col + C], win2, cw, cb)) and torch.equal(win, win2)


@pytest.mark.parametrize("K", [128, 384, 512])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("M,N,col,C,taps", [(64, 3104, 1024, 1024, 4), (40, 1040, 16, 1000, 4), (9, 70, 5, 60, 3)])
def test_conv_step_with_four_waves_and_without_a_norm(M, N, col, C, taps, norm, K):
    """K not a multiple of 256 (four waves to a workgroup), at 64, 32 and 16 rows per workgroup, with and without the
    norm weight, through the C entry: equal bits to the product and the step in their own launches."""
    from cdssm_hip import _lib
    from cdssm_hip.lm import conv1d_silu_step, skinny_linear
    g = torch.Generator().manual_seed(K + N)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)

    x, w, b, nw = rnd(M, K), rnd(N, K), rnd(N), rnd(K) if norm else None
    cw, cb, win = rnd(C, taps), rnd(C), rnd(M, taps - 1, C)
    y, yc, win2 = rnd(M, N), rnd(M, C), win.clone()
    _lib.check(_lib.load().cdssm_skinny_gemm_conv_step(
        1, _lib.ptr(x), K, _lib.ptr(w), K, _lib.ptr(b), _lib.ptr(nw), 1e-5, _lib.ptr(y), N, M, N, K, col,
        _lib.ptr(win), _lib.ptr(cw), _lib.ptr(cb), _lib.ptr(yc), C, taps, _lib.stream_of(DEV)), "conv step")
    want = skinny_linear(x, w, b, norm_weight=nw, eps=1e-5)
    assert torch.equal(y, want)
    assert torch.equal(yc, conv1d_silu_step(want[:, col:col + C], win2, cw, cb)) and torch.equal(win, win2)
