"""The one-launch forward folds the state entering a segment from the maps of the earlier ones with stated
roundings (map_apply in csrc/fwd_lookback.hpp), so that its bits do not depend on how the compiler groups
the multiply-adds.  The gate-level form is given chunk maps that are exact in fp32: per segment of four
chunks one transition g that is not 1 and one written token, so the segment's map is h -> g h + w k, w k an
exact product.  The final state then has to equal the fold restated here, bit for bit.
"""

import numpy as np
import pytest
import torch

from _gpu_util import DEV, log

pytestmark = pytest.mark.gpu

GROUP, ANCHOR, DIRECT, CHUNKS = 8, 64, 15, 4  # segments to a group, to an anchor, folded one by one; chunks to a segment


def fma(a, b, c):
    """a b + c of float32 arrays, rounded once: the product is exact in float64, the sum is rounded to odd
    there, which a later rounding to float32 does not see."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    p, c = np.broadcast_arrays(p, c)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    odd = np.where((s.view(np.int64) & 1) == 0, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
    return np.where(err != 0, odd, s).astype(np.float32)


def apply(g, s, f, im_re):
    gx, gy, sx, sy = g[0], g[1], s[0], s[1]
    re = fma(gx, sx, -(gy * sy))
    im = fma(gy, sx, gx * sy) if im_re else fma(gx, sy, gy * sx)
    return np.stack([re + f[0], im + f[1]])


def product(g, h):
    return np.stack([fma(g[0], h[0], -(g[1] * h[1])), fma(g[0], h[1], g[1] * h[0])])


def fold(G, F, h0, im_re):
    """The final state: G, F (segments, 2, ...) the maps, oldest first; h0 the state entering the first one."""
    n = len(G)

    def entering(seg):
        if seg == 0:
            return h0
        anc = ANCHOR * ((seg - 1) // ANCHOR)
        s = h0 if anc == 0 else leaving(anc - 1)
        maps = []
        first = anc if seg - anc <= DIRECT else seg // GROUP * GROUP
        for g0 in range(anc, first, GROUP):
            Gg, Fg = np.stack([np.ones_like(G[0][0]), np.zeros_like(G[0][0])]), np.zeros_like(F[0])
            for u in range(g0, g0 + GROUP):
                Fg, Gg = apply(G[u], Fg, F[u], im_re), product(G[u], Gg)
            maps.append((Gg, Fg))
        maps += [(G[u], F[u]) for u in range(first, seg)]
        for u, (g, f) in enumerate(maps):
            s = apply(g, s, f, im_re and u > 0)
        return s

    def leaving(seg):
        return apply(G[seg], entering(seg), F[seg], im_re)

    return leaving(n - 1)


# im_re: a thread of the workgroup folds two elements of the state (8 heads of 64 dims, 4 of 128 to a wave)
@pytest.mark.parametrize("dtype,H,D,segments,im_re", [
    (torch.bfloat16, 4, 64, 3, True), (torch.bfloat16, 6, 64, 6, False), (torch.bfloat16, 4, 64, 15, True),
    (torch.bfloat16, 5, 64, 27, False), (torch.bfloat16, 3, 128, 9, True), (torch.bfloat16, 2, 128, 33, True),
    (torch.float32, 3, 64, 4, False), (torch.float32, 2, 128, 21, False), (torch.bfloat16, 3, 64, 70, True)])
@pytest.mark.parametrize("train", [False, True])
def test_final_state_is_the_stated_fold(dtype, H, D, segments, im_re, train):
    from cdssm_hip import check_lookback, set_forward_path
    from cdssm_hip.scan import chunkwise_delta_scan_abar_fwd
    log(f"[carry order] {dtype} H{H} D{D} {segments} segments train={train}")
    g = torch.Generator().manual_seed(segments)
    n = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    L, step = segments * CHUNKS * D, CHUNKS * D
    A, v, k = torch.zeros(1, L, H, 2, dtype=dtype), torch.zeros(1, L, H, 2, dtype=dtype), torch.zeros(1, L, H, D, dtype=dtype)
    A[..., 0] = 1
    # rotations a little inside the unit disc: every map of the fold reaches the result
    turn = 3 * torch.rand(segments, H, generator=g)
    size = 0.9 + 0.1 * torch.rand(segments, H, generator=g)
    A[0, ::step] = torch.stack([size * turn.cos(), size * turn.sin()], -1).to(dtype)
    # bf16 values, so that the written w k is an exact product also where the tensors are fp32
    v[0, step - 1::step], k[0, step - 1::step] = n(segments, H, 2).bfloat16().to(dtype), n(segments, H, D).bfloat16().to(dtype)
    one = torch.ones(1, L, H, dtype=dtype)
    h0 = torch.randn(1, H, 2, D, generator=g)
    x = [t.to(DEV) for t in (n(1, L, H, D), k, v, one, one, A, one[..., None].contiguous())]
    prev = set_forward_path("one_pass")
    try:
        h = chunkwise_delta_scan_abar_fwd(*x, h0=h0.to(DEV), train=train)[1].cpu().numpy()[0]
    finally:
        set_forward_path(prev)
    check_lookback()
    G = A[0, ::step].float().numpy().transpose(0, 2, 1)[..., None]                   # (segments, 2, H, 1)
    F = (v[0, step - 1::step].float()[..., None] * k[0, step - 1::step].float()[:, :, None]).numpy()
    ref = fold(G, F.transpose(0, 2, 1, 3), h0[0].numpy().transpose(1, 0, 2), im_re)  # (2, H, D)
    assert np.array_equal(h.transpose(1, 0, 2), ref), np.abs(h.transpose(1, 0, 2) - ref).max()
