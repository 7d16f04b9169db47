"""Which whole-call decodes the chunk kernel takes, and how it cuts them (the host's
rule and a model of the device's search, kivi_decode_mfma.hip plan_chunks and
chunk_units): a call that some mix of lengths makes slower there than in the stream goes
to the stream, and whatever the lengths, no chunk is left without a workgroup."""
from __future__ import annotations

import ctypes
import random

import pytest

from jacq_amd import kivi

CUS = 256


def plan(nh, nkv, hd, page, R, batch, tokens, per_query=0, cus=CUS):
    geo = kivi.Geometry(nh, nkv, hd, page, 32, R, tokens // page, 1 << 20)
    out = (ctypes.c_int32 * 5)()
    kivi.lib().jacq_kivi_test_plan_decode(ctypes.byref(geo), batch, ctypes.c_int64(tokens),
                                          per_query, cus, out)
    return dict(zip(("waves", "grid", "slots", "units", "whole"), out))


# (heads, batch, longest): 3 to 36% slower in the chunk kernel for the lengths named
@pytest.mark.parametrize("nh,nkv,hd,page,batch,tokens", [
    (40, 8, 128, 16, 17, 16000),  # equal lengths: one workgroup on 136 of 256 CUs
    (40, 8, 128, 16, 17, 8400), (40, 8, 128, 16, 11, 30000),  # equal
    (40, 8, 128, 16, 11, 40000),  # equal: two on 88
    (40, 8, 128, 16, 20, 14000),  # 13 long ones among 7 short
    (40, 8, 128, 16, 72, 1376), (40, 8, 128, 16, 72, 512),   # 25 long ones
    (40, 8, 128, 16, 96, 2752),   # a single long one
    (32, 2, 128, 32, 132, 5632),  # 125 long ones
    (14, 2, 64, 16, 44, 32000), (14, 2, 64, 16, 132, 4000), (14, 2, 64, 16, 192, 300),
    (14, 2, 64, 16, 128, 4000),   # a single long one
])
def test_calls_a_mix_of_lengths_slows_take_the_stream(nh, nkv, hd, page, batch, tokens):
    assert plan(nh, nkv, hd, page, 128, batch, tokens)["waves"] == 0


@pytest.mark.parametrize("nh,nkv,hd,page,R,batch,tokens", [
    (40, 8, 128, 16, 128, 1, 262144), (40, 8, 128, 16, 128, 8, 65536),
    (40, 8, 128, 16, 128, 17, 4000), (32, 8, 128, 16, 128, 32, 4128),
    (40, 8, 128, 16, 128, 96, 192), (32, 2, 128, 32, 128, 80, 6016),
    (14, 2, 64, 16, 128, 16, 32768), (32, 4, 64, 16, 32, 1, 262144), (14, 2, 64, 16, 32, 256, 64)])
def test_calls_faster_in_chunks_whatever_the_lengths(nh, nkv, hd, page, R, batch, tokens):
    assert plan(nh, nkv, hd, page, R, batch, tokens)["waves"] > 0


def device_chunks(units, nkv, p):
    """chunk_units() and chunk_count(): the call's chunks, and units per chunk."""
    count = lambda cu: nkv * sum(1 if u <= p["whole"] else -(-u // cu) for u in units)
    slots = max(p["slots"], len(units) * nkv)
    lo = max(p["units"], -(-sum(units) * nkv // slots))
    if count(lo) <= slots:
        return count(lo)
    hi = 2 * lo
    while count(hi) > slots:
        lo, hi = hi, 2 * hi
    while hi - lo > lo // 16 + 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if count(mid) <= slots else (mid, hi)
    return count(hi)


def test_every_chunk_has_a_workgroup_and_a_workspace_slot():
    rng = random.Random(2)
    taken = 0
    for _ in range(4000):
        nh, nkv, hd = rng.choice([(40, 8, 128), (32, 2, 128), (14, 2, 64), (8, 1, 64), (32, 4, 64),
                                  (8, 8, 128), (16, 1, 128)])
        R, batch = rng.choice([32, 64, 128, 256]), int(2 ** rng.uniform(0, 8.1))
        tokens = int(2 ** rng.uniform(4, 17)) // 32 * 32 + R
        p = plan(nh, nkv, hd, 16, R, batch, tokens, cus=rng.choice([CUS, 64, 304]))
        if not p["waves"]:
            continue
        taken += 1

        def units(n):
            old = max(0, n - R) // 32
            return old + 3 * max(1 if n <= R else 0, -(-(n - 32 * old) // 32))
        long = rng.randint(0, batch)
        lens = [tokens if i < long else rng.randint(0, tokens if rng.random() < .5 else 64)
                for i in range(batch)]
        n = device_chunks([units(x) for x in lens], nkv, p)
        assert n <= p["grid"] <= max(p["slots"], batch * nkv)
    assert taken > 500


def test_bench_names_the_kernel_that_runs():
    import bench
    for (nh, nkv, hd, batch, pages), want in (((40, 8, 128, 64, 1024), "stream"),
                                              ((32, 8, 128, 32, 256), "chunk"),
                                              ((32, 4, 64, 1, 40), "chunk")):
        geo = kivi.KiviGeometry(nh, nkv, hd, 16, 32, 128, pages, 1 << 16)
        assert bench.decode_kernel(kivi, geo, batch, CUS) == want
