"""Appends that age several groups out in one launch, from every kind of
start: an empty cache, a scratch that ends inside or at the edge of a 32-token
group, and one with a group about to age out.  Groups with a scratch row go
through the scratch's wavefronts, groups of new tokens alone through their own,
so the counts lie around the window R, where the second kind begins, and around
whole groups.  Pages and live scratch rows equal the oracle's token-by-token
writes bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from jacq_amd import workloads as wl
from tests.kivi_testlib import State, to_torch

torch = pytest.importorskip("torch")

POOL = ("k_code", "k_scale", "k_zero", "v_code", "v_scale", "v_zero")


def _bits(t):
    t = t.detach().cpu()
    return (t.view(torch.int16) if t.dtype == torch.float16 else t).numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,hd,page,R", [(8, 2, 128, 16, 128), (6, 3, 64, 32, 64),
                                              (5, 1, 128, 32, 32), (4, 2, 64, 16, 256)])
@pytest.mark.parametrize("more", [-1, 0, 1, 31, 32, 33, 77, 160])
def test_append_from_every_kind_of_start(nh, nkv, hd, page, R, more):
    from jacq_amd import kivi
    n = R + more
    starts = [0, 1, 31, 32, R - 1, R, R + 1, R + 31, R + 32, 3 * R + 45]
    w = wl.Workload("span", nh, nkv, hd, len(starts), 1, 1, page=page, residual=R, outliers=2,
                    outlier_scale=9.0, seed=41)
    st = State(w, lens=starts, extra_tokens=n, seed=97 + more)
    st.build_oracle()
    geo = kivi.KiviGeometry(nh, nkv, hd, page, 32, R, st.max_pages, st.num_pages)
    cache = kivi.PagedKiviCache.from_tensors(geo, to_torch(st))
    new = [torch.from_numpy(np.stack([h[b][s:s + n] for b, s in enumerate(starts)])).view(
        torch.float16).cuda() for h in (st.k_hist, st.v_hist)]
    cache.append(*new, torch.from_numpy(st.tables).cuda(),
                 torch.tensor(starts, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    ends = [s + n for s in starts]
    _go_on(st, starts, ends)
    for name in POOL:
        got, want = _bits(getattr(cache, name)), getattr(st.cache, name)
        assert np.array_equal(got.view(want.dtype), want), (name, n)
    for name in ("k_scr", "v_scr"):
        got, want = _bits(getattr(cache, name)).view(np.uint16), getattr(st.cache, name)
        for b, e in enumerate(ends):
            live = e - wl.split_old_tokens(e, R)
            assert np.array_equal(got[b, :, :live], want[b, :, :live]), (name, n, starts[b])


def _go_on(st, starts, ends):
    from oracle import oracle as o
    for b, (s, e) in enumerate(zip(starts, ends)):
        for t in range(s, e):
            o.cache_write(st.cache, b, st.k_hist[b][t], st.v_hist[b][t], st.tables[b], t + 1)


def test_code_by_reciprocal_equals_division():
    """The writer takes rint((x - min) * rcp(scale)) where that lies further
    than 2^-16 from a rounding boundary and divides elsewhere: with any
    reciprocal within 1 ulp, every code it takes is the division's, over fp16
    tiles of every exponent and quotients placed at the boundaries."""
    rng = np.random.default_rng(7)
    f = np.float32
    bits = rng.integers(0, 1 << 16, (200_000, 2), dtype=np.uint16)
    ends = np.sort(bits.view(np.float16).astype(f), 1)
    ends = ends[np.isfinite(ends).all(1)]
    mn, mx = ends.T
    s = (mx - mn) / f(15)
    s = np.where(s > 0, s, f(1))
    at = rng.integers(0, 31, mn.size).astype(f) / f(2)  # whole and half codes
    near = at + rng.choice([0.0, 1e-6, -1e-6, 1e-4, -1e-4, 0.2], mn.size).astype(f)
    x = np.clip((mn + near * s).astype(np.float16).astype(f), mn, mx)
    exact = np.clip(np.rint((x - mn) / s), 0, 15)
    taken = 0
    for inv in (np.nextafter(f(1) / s, f(0)), f(1) / s, np.nextafter(f(1) / s, f(np.inf))):
        q = (x - mn) * inv
        sure = np.abs(q - np.rint(q)) < f(0.5 - 2 ** -16)
        assert np.array_equal(np.rint(q)[sure], exact[sure])
        taken += sure.mean() / 3
    assert taken > 0.5
