"""GPU parity of the matrix-core one-launch forward (the bf16 scan-level inference forward where one round of
workgroups holds every segment) at the sizes where its blocks, chunks and head groups end, against the
fp64 oracle on the same rounded inputs.

Tolerances: y is rounded once to bf16, 2^-9 of the value, so 2^-8 of the largest value leaves as much
again for the sums; the state is fp32 throughout with operands split to 2^-24, the dynamics' hardware
log / exp (2e-5) being the largest error, so 5e-5 of the largest state value.
"""

import pytest
import torch

from _gpu_util import DEV, ScanConfig, draw_inputs, log, on_matrix_cores, oracle_fwd, rel, select, to_dev

pytestmark = pytest.mark.gpu

TOL_Y, TOL_H = 2.0 ** -8, 5e-5
KEYS = ("q", "k", "v", "beta", "sel_C", "dt", "r", "alpha", "omega")


def run(x, chunk=None):
    from cdssm_hip import check_lookback, chunkwise_delta_scan
    B, L, H, D = x["q"].shape
    assert on_matrix_cores(ScanConfig("t", B=B, H=H, L=L, D=D))
    y, h = chunkwise_delta_scan(*[x[n] for n in KEYS], x["c"], h0=x.get("h0"), chunk_size=chunk)
    torch.cuda.synchronize()
    check_lookback()
    return y.cpu(), h.cpu()


@pytest.mark.parametrize("B,H,L,D,chunk", [
    (1, 1, 1, 64, None), (2, 3, 15, 64, None), (1, 4, 16, 64, None), (1, 5, 17, 64, None), (1, 8, 64, 64, None),
    (3, 6, 65, 64, None), (1, 4, 257, 64, None), (2, 7, 100, 64, 1), (1, 4, 130, 64, 17), (1, 6, 300, 64, 128),
    (1, 2, 1, 128, None), (2, 5, 127, 128, None), (1, 4, 513, 128, None), (1, 3, 200, 128, 48)])
def test_matches_oracle_at_the_edges_of_blocks_chunks_and_head_groups(B, H, L, D, chunk):
    log(f"[mfma forward] B{B} H{H} L{L} D{D} chunk={chunk or D}")
    x = draw_inputs(ScanConfig("t", B=B, H=H, L=L, D=D, h0_std=0.1), seed=L + H)
    y, h = run(to_dev(x), chunk)
    yr, hr = oracle_fwd(x, chunk)
    assert rel(y, yr) <= TOL_Y and rel(h, hr) <= TOL_H, (rel(y, yr), rel(h, hr))


@pytest.mark.parametrize("D,segments", [(64, 15), (64, 17), (64, 70), (128, 66)])
def test_matches_oracle_over_group_and_anchor_ends(D, segments):
    """More segments than are folded one by one (15), than one group, and than lie between two anchors (64): heads
    with a slow decay, so that a state entering the first segments reaches the last ones.  Its factor is a product of
    L transitions, each formed in fp32 with a hardware reciprocal and exponential: off by 2^-23 each, L 2^-23 in
    all; a map folded twice or not at all is wrong by the values' size."""
    log(f"[mfma forward] {segments} segments D{D}")
    x = draw_inputs(ScanConfig("t", B=2, H=4, L=segments * 4 * D - 5, D=D, h0_std=1.0), seed=segments)
    x["alpha"], x["omega"], x["r"] = x["alpha"] * 1e-4, x["omega"] * 1e-3, x["r"] * 1e-3
    y, h = run(to_dev(x))
    yr, hr = oracle_fwd(select(x, [1], [2]))
    ey, eh, tol = rel(y[1:2, :, 2:3], yr), rel(h[1:2, 2:3], hr), x["q"].shape[1] * 2.0 ** -23
    assert ey <= TOL_Y + tol and eh <= TOL_H + tol, (ey, eh, tol)


@pytest.mark.parametrize("alpha,omega", [(3.0, 0.02), (1.0, 0.0), (10.0, 0.1)])
@pytest.mark.parametrize("D", [64, 128])
def test_strong_decay_runs_blocks_in_true_units(D, alpha, omega):
    """|a_t| far below 2^-5: the products of a over 16 tokens underflow their reciprocal, so most blocks run
    the true-units solve."""
    log(f"[mfma forward] strong decay D{D} alpha x{alpha} omega x{omega}")
    x = draw_inputs(ScanConfig("t", B=1, H=6, L=300, D=D, h0_std=0.1), seed=3)
    x["alpha"], x["omega"] = x["alpha"] * alpha, x["omega"] * omega
    y, h = run(to_dev(x))
    yr, hr = oracle_fwd(x)
    assert rel(y, yr) <= TOL_Y and rel(h, hr) <= TOL_H, (rel(y, yr), rel(h, hr))


def test_misaligned_scalars_take_the_element_loads():
    """beta, sel_C, dt, r and v one element off their 8-byte (4-byte) alignment: the same values, bit for bit."""
    x = to_dev(draw_inputs(ScanConfig("t", B=2, H=8, L=333, D=64), seed=1))
    ref = run(x)
    for n in ("v", "beta", "sel_C", "dt", "r"):
        t = torch.empty(x[n].numel() + 1, dtype=x[n].dtype, device=DEV)[1:].view(x[n].shape)
        x[n] = t.copy_(x[n])
        assert x[n].data_ptr() % 4 == 2
    got = run(x)
    assert torch.equal(ref[0], got[0]) and torch.equal(ref[1], got[1])


@pytest.mark.parametrize("name,value", [("k", float("nan")), ("k", float("inf")), ("q", float("nan")),
                                        ("v", float("inf")), ("dt", float("nan"))])
def test_non_finite_input_stays_in_its_head(name, value):
    """One non-finite element in head 1 at token 37: the other heads of the wave are bit-identical to a clean
    run's, head 1 is so before that token and non-finite at it (q: at it only)."""
    B, H, L, t, h = 1, 4, 150, 37, 1
    log(f"[mfma forward] {value} in {name}")
    x = to_dev(draw_inputs(ScanConfig("t", B=B, H=H, L=L, D=64), seed=2))
    y0, h0 = run(x)
    x[name] = x[name].clone()
    x[name][0, t, h].view(-1)[0] = value
    y1, h1 = run(x)
    rest = [i for i in range(H) if i != h]
    assert torch.equal(y0[:, :, rest], y1[:, :, rest]) and torch.equal(h0[:, rest], h1[:, rest])
    assert torch.equal(y0[:, :t, h], y1[:, :t, h])
    assert not y1[:, t, h].isfinite().any()
    if name == "q":
        assert torch.equal(y0[:, t + 1:, h], y1[:, t + 1:, h]) and torch.equal(h0, h1)
    else:
        assert not y1[:, -1, h].isfinite().any() and not h1[:, h].isfinite().any()


def test_continuing_call_after_a_four_launch_training_call():
    """A *_continue inference call on a workspace whose previous call was a training forward of the shape, which
    takes four launches here (more segments of 8 heads than compute units): the look-back epoch is there."""
    from cdssm_hip import _lib, check_lookback
    from cdssm_hip.scan import PreparedForward
    x = to_dev(draw_inputs(ScanConfig("t", B=1, H=20, L=64 * 4 * 90, D=64), seed=4))
    args = [x[n] for n in KEYS]
    train, infer = PreparedForward(*args, x["c"], train=True), PreparedForward(*args, x["c"])
    infer()
    torch.cuda.synchronize()
    y, h = infer.y.clone(), infer.h_final.clone()
    train()
    a = list(infer._args)
    a[-7] = _lib.ptr(train.workspace)
    for _ in range(3):
        infer.y.zero_()
        st = infer._lib.cdssm_fused_scan_fwd_continue(*a, _lib.stream_of(DEV))
        assert st == 0
        torch.cuda.synchronize()
        check_lookback()
        assert torch.equal(infer.y, y) and torch.equal(infer.h_final, h)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("source", ["carried", "written"])
def test_a_large_state_that_is_overwritten_leaves_fp32_accuracy(source, D):
    """Tokens with beta near 1 erase a state S times the values written over it, and the readout asks for the
    direction just erased: y is what is left of two parts of size S.  Beside y's own rounding, half a bf16 ulp, its
    error is that of fp32 sums of such parts, 2^-22 of their size (a few roundings of 2^-24; a state projects on a
    direction with up to 4 S); operands of two bf16 terms would leave 2^-17.  alpha = omega = 0 and a small r, so that the transitions are 1 to 1e-7 and vp its clamp,
    1e-3, and the dynamics' own error stays relative to y."""
    log(f"[mfma forward] overwritten {source} D{D}")
    B, H, L, S = 2, 5, 64, 100.0
    g = torch.Generator().manual_seed(D)
    n = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
    pool = unit(n(B, 1, H, 6, D)).expand(B, L, H, 6, D)
    pick = lambda t: torch.gather(pool, 3, t[..., None, None].expand(B, L, H, 1, D))[:, :, :, 0]  # noqa: E731
    ki = torch.randint(0, 6, (B, L, H), generator=g)
    # the correction is read before the token's erasure, the local state after it
    qi = torch.roll(ki, 1, 1) if source == "carried" else ki
    size = torch.ones(L) if source == "carried" else torch.where(torch.arange(L) % 32 < 8, S, 1.0)
    full = lambda v: torch.full((B, L, H), v)  # noqa: E731
    x = dict(q=pick(qi), k=pick(ki), v=1e3 * n(B, L, H, 2) * size[:, None, None], beta=full(0.996), sel_C=full(1.0),
             dt=full(0.5), r=full(0.05))
    x = {name: t.to(torch.bfloat16).contiguous() for name, t in x.items()}
    x.update(alpha=torch.zeros(H), omega=torch.zeros(H), c=4.0,
             h0=S * n(B, H, 2, D) if source == "carried" else torch.zeros(B, H, 2, D))
    y, h = run(to_dev(x))
    yr, hr = oracle_fwd(x)
    half_ulp = torch.exp2(yr.abs().clamp(min=1e-30).log2().floor() - 8)
    over = ((y.double() - yr).abs() - half_ulp).clamp(min=0).max() / (4 * S)
    log(f"   beyond y's rounding: {float(over):.1e} of the state")
    assert float(over) <= 2.0 ** -22
    assert rel(h, hr) <= TOL_H


def _flat_dynamics(H, E, c, cr):
    """alpha, omega, c, and dt, r, for which every transition is real and |a| = E^(cr / 2)."""
    ta = (1 - E ** 0.5) / (1 + E ** 0.5)  # ((1 - ta) / (1 + ta))^2 = E
    return dict(alpha=torch.full((H,), 2 * ta), omega=torch.zeros(H), c=c), 1.0, cr / c


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("E,cr,size,L", [
    (2.0 ** -9, 1.0, 2.0 ** 60, 130),   # |a| = 2^-4.5: 2^-72 over a block, under writes of 2^60
    (2.0 ** -12, 1.0, 2.0 ** 100, 70),  # 2^-96 and 2^100
    (2.0 ** -6, 1.0, 2.0 ** 90, 130),   # 2^-48 and 2^90
    (2.0 ** -6, -0.9, 1e3, 24),         # |a| = 2^2.7: grows by 2^43 over a block
])
def test_writes_and_transitions_near_the_limits_stay_finite(D, E, cr, size, L):
    """Quotients of a write and the block's product of transitions beyond fp32's range, with every value of the
    recurrence inside it: those blocks run in true units.  The transitions' hardware exponentials are 2e-5 off, and
    24 of them multiply where they grow."""
    log(f"[mfma forward] limits D{D} E{E:.1e} cr{cr} size{size:.0e} L{L}")
    B, H = 2, 6
    rates, dt, r = _flat_dynamics(H, E, 4.0, cr)
    x = draw_inputs(ScanConfig("t", B=B, H=H, L=L, D=D), seed=7)
    x.update(rates, v=x["v"] * size, dt=torch.full_like(x["dt"], dt), r=torch.full_like(x["r"], r), h0=None)
    x = {k: v for k, v in x.items() if v is not None}
    if cr < 0:
        x["v"][:, :12] = 0  # what is written last in the first block, where the product is largest, decides
    y, h = run(to_dev(x))
    yr, hr = oracle_fwd(x)
    assert y.isfinite().all() and h.isfinite().all()
    tol = 24 * 2e-5 if cr < 0 else 0.0
    assert rel(y, yr) <= TOL_Y + tol and rel(h, hr) <= TOL_H + tol, (rel(y, yr), rel(h, hr))


@pytest.mark.parametrize("D", [64, 128])
def test_a_heads_bits_do_not_depend_on_the_others_of_its_wave(D):
    """Heads beside one that decays fast, so that its blocks run in true units, or that holds a NaN in its last
    block: the same bits as beside an ordinary one."""
    log(f"[mfma forward] neighbours D{D}")
    x = to_dev(draw_inputs(ScanConfig("t", B=2, H=8, L=333, D=D, h0_std=0.1), seed=11))
    ref = run(x)
    rest = [0, 1, 3, 4, 5, 7]
    for change in ("decay", "dt", "k", "h0"):
        z = {n: (t.clone() if isinstance(t, torch.Tensor) else t) for n, t in x.items()}
        if change == "decay":
            z["alpha"][[2, 6]] = 12.0
        elif change == "h0":
            z["h0"][:, [2, 6], 0, 3] = float("nan")
        else:
            z[change][:, 330, [2, 6]] = float("nan")
        y, h = run(z)
        assert torch.equal(y[:, :, rest], ref[0][:, :, rest]) and torch.equal(h[:, rest], ref[1][:, rest]), change
        assert not torch.equal(h[:, [2, 6]], ref[1][:, [2, 6]]), change


@pytest.mark.parametrize("name", ["beta", "k", "v"])
def test_non_finite_input_in_two_heads_of_a_wave(name):
    """Head 0 at token 20, head 3 at token 100, of one wave: each is clean before its token and not finite from it
    on, and the other heads are a clean run's."""
    x = to_dev(draw_inputs(ScanConfig("t", B=1, H=5, L=150, D=64), seed=5))
    y0, h0 = run(x)
    x[name] = x[name].clone()
    for h, t in ((0, 20), (3, 100)):
        x[name][0, t, h] = float("inf")
    y1, h1 = run(x)
    assert torch.equal(y0[:, :, [1, 2, 4]], y1[:, :, [1, 2, 4]]) and torch.equal(h0[:, [1, 2, 4]], h1[:, [1, 2, 4]])
    for h, t in ((0, 20), (3, 100)):
        assert torch.equal(y0[:, :t, h], y1[:, :t, h])
        assert not y1[:, t:, h].isfinite().any() and not h1[:, h].isfinite().any()
