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


GEOMETRIES = pytest.mark.parametrize("nh,nkv,hd,page,R", [
    (8, 2, 128, 16, 128), (6, 3, 64, 32, 64), (5, 1, 128, 32, 32), (4, 2, 64, 16, 256)])


@pytest.mark.gpu
@GEOMETRIES
@pytest.mark.parametrize("more", [-1, 0, 1, 31, 32, 33, 77, 160])
def test_append_from_every_kind_of_start(nh, nkv, hd, page, R, more):
    _append(nh, nkv, hd, page, R, R + more, seed=97 + more)


@pytest.mark.gpu
@GEOMETRIES
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 16, 17, 30])
def test_append_of_few_tokens(nh, nkv, hd, page, R, n):
    """Counts around the rows of a wavefront's load (4 or 8) and of a workgroup's (16)."""
    _append(nh, nkv, hd, page, R, n, seed=197 + n)


def _append(nh, nkv, hd, page, R, n, seed):
    from jacq_amd import kivi
    starts = [0, 1, 31, 32, R - 1, R, R + 1, R + 31, R + 32, 3 * R + 45]
    w = wl.Workload("span", nh, nkv, hd, len(starts), 1, 1, page=page, residual=R, outliers=2,
                    outlier_scale=9.0, seed=41)
    st = State(w, lens=starts, extra_tokens=n, seed=seed)
    st.build_oracle()
    _append_and_compare(kivi, st, starts, n)


def _append_and_compare(kivi, st, starts, n):
    w, R = st.w, st.w.residual
    geo = kivi.KiviGeometry(w.nh, w.nkv, w.hd, w.page, 32, R, st.max_pages, st.num_pages)
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


def _half_code_lines(rng, count):
    """Lines of 32 fp16 values: a minimum, a maximum, the 15 values next to the half codes
    between them and one value beside each of those.  In a quarter of the lines the scale
    is a power of two and the values are the half codes themselves; the others are those of
    many whose values come closest to one."""
    f = np.float32
    lo = rng.uniform(-8, 8, 40 * count).astype(np.float16)
    hi = (lo.astype(f) + rng.uniform(0.5, 20, lo.size).astype(f)).astype(np.float16)
    exact = count // 4
    lo[:exact] = 0
    hi[:exact] = 15 * 2.0 ** rng.integers(-6, 4, exact)
    s = (hi.astype(f) - lo.astype(f)) / f(15)
    half = np.arange(15, dtype=f) + f(0.5)
    x = (lo.astype(f)[:, None] + half * s[:, None]).astype(np.float16)
    off = np.abs((x.astype(f) - lo.astype(f)[:, None]) / s[:, None] - half).min(1)
    pick = np.concatenate([np.arange(exact), exact + np.argsort(off[exact:])[:count - exact]])
    lo, hi, x = lo[pick], hi[pick], x[pick]
    beside = np.nextafter(x, np.where(rng.random(x.shape) < 0.5, -np.inf, np.inf).astype(np.float16))
    lines = np.concatenate([lo[:, None], hi[:, None], x, np.clip(beside, lo[:, None], hi[:, None])], 1)
    return rng.permuted(lines, axis=1)


@pytest.mark.gpu
@pytest.mark.parametrize("hd,start", [(128, 0), (128, 31), (64, 0), (64, 40)])
def test_codes_at_half_codes(hd, start):
    """Quotients on, within 2^-16 of and just past the rounding boundaries, so that the
    reciprocal's codes and the division's both occur, in groups of new tokens and in
    groups that go through the scratch."""
    from jacq_amd import kivi
    nkv, R, groups = 2, 32, 6
    w = wl.Workload("half", nkv, nkv, hd, 1, 1, 1, page=16, residual=R, seed=43)
    n = R + 32 * groups + 32
    st = State(w, lens=[start], extra_tokens=n, seed=5)
    rng = np.random.default_rng(hd + start)
    k = _half_code_lines(rng, groups * nkv * hd).reshape(groups, nkv, hd, 32)  # per channel
    v = _half_code_lines(rng, groups * 32 * nkv * hd // 32)  # per token and 32 channels
    st.k_hist[0][:32 * groups] = k.transpose(0, 3, 1, 2).reshape(-1, nkv, hd).view(np.uint16)
    st.v_hist[0][:32 * groups] = v.reshape(-1, nkv, hd).view(np.uint16)
    f = np.float32
    for x, axis in ((k, 3), (v.reshape(-1, 32), 1)):
        lo, hi = x.min(axis, keepdims=True).astype(f), x.max(axis, keepdims=True).astype(f)
        q = (x.astype(f) - lo) / ((hi - lo) / f(15))
        off = np.abs(q - np.rint(q))
        assert (off >= 0.5 - 2 ** -16).sum() > 100 and (off < 0.5 - 2 ** -16).sum() > 100
        assert ((off < 0.5 - 2 ** -16) & (off > 0.5 - 2 ** -12)).sum() > 20
    st.build_oracle()
    _append_and_compare(kivi, st, [start], n)


def _go_on(st, starts, ends):
    from oracle import oracle as o
    for b, (s, e) in enumerate(zip(starts, ends)):
        for t in range(s, e):
            o.cache_write(st.cache, b, st.k_hist[b][t], st.v_hist[b][t], st.tables[b], t + 1)


def test_code_by_reciprocal_equals_division():
    """The rule that the writer's codes follow (the kernel's own are in
    test_codes_at_half_codes): rint((x - min) * rcp(scale)) where that lies further
    than 2^-16 from a rounding boundary, a division elsewhere.  With any
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
