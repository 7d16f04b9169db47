"""The decode of calls of few or short segments ((sequence, kv head) pairs): a
workgroup per chunk of a segment, folded in LDS and across workgroups.  Lengths
lie around where a segment is cut (three units per wavefront), at the edges of
groups and of the fp16 window, and where the fused step ages a group out of a
cut segment; batches around where the call leaves this kernel and where its
sequences fill more than one window of 64."""
from __future__ import annotations

import numpy as np
import pytest

from jacq_amd import workloads as wl
from oracle import oracle as o
from tests.kivi_testlib import State, assert_close, to_torch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

POOL = ("k_code", "k_scale", "k_zero", "v_code", "v_scale", "v_zero", "k_scr", "v_scr")


def _bits(t):
    t = t.detach().cpu()
    return (t.view(torch.int16) if t.dtype == torch.float16 else t).numpy()


def _check(nh, nkv, hd, page, R, lens, seed):
    """A decode and two fused steps (the first ages a group out wherever a
    length is R + 31 modulo 32), eager and replayed, against the oracle."""
    from jacq_amd import kivi
    w = wl.Workload("chunks", nh, nkv, hd, len(lens), 1, 1, page=page, residual=R, outliers=2,
                    outlier_scale=9.0, seed=3)
    st = State(w, lens=lens, extra_tokens=2, seed=seed)
    st.build_oracle()
    geo = kivi.KiviGeometry(nh, nkv, hd, page, 32, R, st.max_pages, st.num_pages)
    cache = kivi.PagedKiviCache.from_tensors(geo, to_torch(st))
    q = torch.from_numpy(st.q).view(torch.float16).cuda()
    bt = torch.from_numpy(st.tables).cuda()
    n = torch.from_numpy(st.lens.astype(np.int32)).cuda()
    out = cache.decode(q, n, bt)
    assert_close(out.cpu().numpy(), st.decode_ref(), "decode")
    graph, again = torch.cuda.CUDAGraph(), torch.empty_like(out)
    with torch.cuda.graph(graph):
        cache.decode(q, n, bt, out=again)
    for _ in range(3):  # the flags are clear after each replay
        again.fill_(3.0)
        graph.replay()
        assert torch.equal(again.view(torch.int32), out.view(torch.int32))
    cur = st.lens.copy()
    for _ in range(2):
        new = [torch.from_numpy(np.stack([h[b][cur[b]] for b in range(len(lens))])).view(
            torch.float16).cuda() for h in (st.k_hist, st.v_hist)]
        out = cache.write_decode(q, *new, torch.from_numpy((cur + 1).astype(np.int32)).cuda(), bt)
        for b in range(len(lens)):
            o.cache_write(st.cache, b, st.k_hist[b][cur[b]], st.v_hist[b][cur[b]], st.tables[b],
                          int(cur[b]) + 1)
        cur = cur + 1
        torch.cuda.synchronize()
        for name in POOL:
            want = getattr(st.cache, name)
            assert np.array_equal(_bits(getattr(cache, name)).view(want.dtype), want), name
        assert_close(out.cpu().numpy(), st.decode_ref(cur), "fused step")


@pytest.mark.parametrize("nh,nkv,hd,page,R", [(10, 2, 128, 16, 128), (32, 2, 128, 32, 64),
                                              (7, 1, 64, 16, 32), (24, 2, 64, 32, 128)])
def test_lengths_around_the_cut(nh, nkv, hd, page, R):
    whole = 24 if hd == 128 and nh // nkv > 8 else 36  # units of a segment kept whole
    groups = whole - 3 * (R // 32)
    edge = R + 32 * groups  # this many units, and one token more starts a residual tile
    _check(nh, nkv, hd, page, R, [edge - 1, edge, edge + 1, edge + 31, edge + 32, R + 31, R + 32,
                                  R - 1, 31, 1, 2 * edge + 31, 12 * edge + 31], seed=nh)


@pytest.mark.parametrize("batch,nkv", [(128, 2), (129, 2), (64, 4), (256, 1), (257, 1), (193, 1),
                                       (96, 8), (97, 8)])
def test_batches_around_the_rules_segment_counts(batch, nkv):
    lens = [1 + (37 * i) % 190 for i in range(batch)]
    lens[::7] = [63 + 32 * (i % 40) for i in range(len(lens[::7]))]
    _check(2 * nkv, nkv, 64, 16, 32, lens, seed=batch)


def test_one_long_sequence_among_short_ones():
    lens = [20, 150, 9000, 159, 33, 700]
    _check(40, 8, 128, 16, 128, lens, seed=5)


def test_v1_queries_of_two_launches_equal_single():
    """160 causal queries of one 4096-token sequence need two launches of a v1
    workspace region; each equals its own jac_launch bit for bit."""
    from jacq_amd import kivi
    w = wl.Workload("v1", 40, 8, 128, 1, 4096, 4096, page=32, residual=128, outliers=8, seed=11)
    st = State(w, lens=[4096], seed=8)
    st.build_oracle()
    g = to_torch(st)
    bt = torch.from_numpy(st.tables[0]).cuda()
    pool = [g[n] for n in POOL[:6]] + [g["k_scr"][0], g["v_scr"][0]]
    seq = np.arange(4096 - 159, 4097).astype(np.int32)
    seq[:4] = [1, 129, 160, 1000]
    q = torch.from_numpy(np.random.default_rng(3).standard_normal((160, 40, 128)).astype(
        np.float16)).cuda()
    out = torch.empty((160, 40, 128), dtype=torch.float32, device="cuda")
    kivi.kivi_decode_batched_dsl(q, torch.from_numpy(seq).cuda(), bt, *pool, 160, out)
    one = torch.empty((40, 128), dtype=torch.float32, device="cuda")
    for i in list(range(0, 160, 13)) + [1, 2, 3, 88, 89, 90, 159]:
        kivi.kivi_decode_dsl(q[i].contiguous(), bt, *pool, int(seq[i]), one)
        assert torch.equal(one.view(torch.int32), out[i].view(torch.int32)), i


@pytest.mark.parametrize("nh,nkv,hd,page", [(10, 2, 128, 16), (32, 2, 128, 32), (14, 2, 64, 16),
                                            (20, 2, 64, 32)])
def test_one_tile_sequences_equal_the_stream(nh, nkv, hd, page):
    """A sequence of up to 32 tokens is one wavefront's, which writes O from its registers in
    both kernels: the same bits, beside longer sequences and with none."""
    from jacq_amd import kivi
    for lens in ([0, 1, 31, 32], [32, 33, 200, 7, 1000]):
        w = wl.Workload("short", nh, nkv, hd, len(lens), 1, 1, page=page, residual=64, outliers=2,
                        outlier_scale=9.0, seed=5)
        st = State(w, lens=lens, seed=hd)
        st.build_oracle()
        geo = kivi.KiviGeometry(nh, nkv, hd, page, 32, 64, st.max_pages, st.num_pages)
        cache = kivi.PagedKiviCache.from_tensors(geo, to_torch(st))
        q = torch.from_numpy(st.q).view(torch.float16).cuda()
        args = (q, torch.from_numpy(st.lens.astype(np.int32)).cuda(),
                torch.from_numpy(st.tables).cuda())
        chunk = cache.decode(*args)
        kivi.lib().jacq_kivi_test_force_stream(1)
        try:
            stream = cache.decode(*args)
        finally:
            kivi.lib().jacq_kivi_test_force_stream(0)
        assert_close(chunk.cpu().numpy(), st.decode_ref(), "decode")
        for b, n in enumerate(lens):
            if n <= 32:
                assert torch.equal(chunk[b].view(torch.int32), stream[b].view(torch.int32)), n
