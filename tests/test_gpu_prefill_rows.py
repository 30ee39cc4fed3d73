"""fp32 prefill computes every query row from the row and the keys it attends alone: the same bits whichever rows
share its workgroup, whichever sequences its call and wherever the prompt is cut, at f32 precision, for data that the
f16 pieces cannot hold (infinities, NaN, wide spreads) beside data that they can."""
from __future__ import annotations

import numpy as np
import pytest

from glint_amd import synth
from gpu_util import Contig, run_prefill
from helpers import attention_f64

pytestmark = pytest.mark.gpu


def _same(a, b):
    """Equal bits; any NaN equals any NaN."""
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    return np.array_equal(np.where(np.isnan(a), np.uint32(0x7FC00000), a.view(np.uint32)),
                          np.where(np.isnan(b), np.uint32(0x7FC00000), b.view(np.uint32)))


def _plant(what, at, k, v, q):
    """One sequence's data [n][Hkv*d] and rows [n][H][d] with something odd at position `at`."""
    if what == "q_inf":
        q[at, 1, 3] = np.inf
    elif what == "q_spread":  # eight dims far below the row's others
        q[at, :, 8:16] *= np.float32(2.0**-40)
    elif what == "k_inf":
        k[at, 5] = -np.inf
    elif what == "k_spread":
        k[at, 8:16] *= np.float32(2.0**-30)
    elif what == "k_large":
        k[at] *= np.float32(300.0)
    elif what == "v_nan":
        v[at, 7] = np.nan
    elif what == "v_inf":
        v[at, 7], v[at + 3, 9] = np.inf, -np.inf
    elif what == "v_large":
        v[at] *= np.float32(3e4)
    elif what == "v_small":
        v[at:at + 20] *= np.float32(2.0**-18)
    elif what == "v_spread":  # one run small beside the rest of a tile: 2^-14, then 2^-30
        v[at, ::16] *= np.float32(2.0**-14)
        v[at + 1, 1::16] *= np.float32(2.0**-30)
    elif what == "sink":  # the first key's K large and its V small, the next ones' V smaller yet
        k[0] *= np.float32(100.0)
        v[0] *= np.float32(2.0**-9)
        v[1:40] *= np.float32(2.0**-17)
    elif what == "v_tiny":  # rows that attend only these have outputs of 2^-100
        v[:64] *= np.float32(2.0**-100)
    elif what == "v_zero":
        v[at:at + 40] = 0.0
    elif what == "v_max":  # bf16 would round it to infinity; the output is finite
        v[at, 3] = np.float32(3.4e38)


WHAT = ["q_inf", "q_spread", "k_inf", "k_spread", "k_large", "v_nan", "v_inf", "v_large", "v_small", "v_spread",
        "sink", "v_tiny", "v_zero", "v_max"]


@pytest.mark.parametrize("dtype", ["f32", "q8"])
@pytest.mark.parametrize("what", WHAT)
def test_rows_do_not_depend_on_their_neighbours(backend, dtype, what):
    """A prompt alone (one 16-query tile per wave), in a batch that fills the chip (two), and in pieces that are cut
    inside a 32-key tile and short enough to convert their own tiles: the same bits for every row."""
    d, H, Hkv, n, at = 128, 8, 2, 900, 371
    lens = [n] + [n - 1] * 7
    k = synth.normal_rows(61, 8 * n, Hkv * d).reshape(8, 1, n, Hkv * d)
    v = synth.normal_rows(62, 8 * n, Hkv * d).reshape(8, 1, n, Hkv * d)
    q = synth.normal(63, (sum(lens), H, d))
    _plant(what, at, k[0, 0], v[0, 0], q[:n])
    c = Contig(backend, dtype, 8, 1, n, Hkv, d, k=k, v=v)
    start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    slot = np.array([0], np.int32)
    for window in (None, 333):
        both = run_prefill(backend, c.cache, q, start, [0] * 8, H, 0.09, None, window)[:n]
        alone = run_prefill(backend, c.cache, q[:n], [0, n], [0], H, 0.09, None, window, seq_slot=slot)
        assert _same(alone, both), (what, window, "alone")
        for cuts in ([0, at - 3, at + 5, n], [0, 30, 62, 160, 256, 340, at, at + 1, at + 30, 500, 596, n]):
            got = [run_prefill(backend, c.cache, q[a:b], [0, b - a], [a], H, 0.09, None, window, seq_slot=slot)
                   for a, b in zip(cuts, cuts[1:])]
            assert _same(np.concatenate(got), both), (what, window, cuts)


@pytest.mark.parametrize("dtype", ["f32", "q8"])
@pytest.mark.parametrize("d,H,Hkv", [(64, 9, 3), (128, 8, 2), (256, 4, 2)])
def test_workgroups_that_convert_give_the_staged_bits(backend, d, H, Hkv, dtype):
    """A storage of three tiles: a prompt of all its rows is staged, one in pieces of up to 32 rows converts its
    tiles in the workgroups."""
    n = 96
    for at in (0, 37, 60):
        for what in WHAT:
            k = synth.normal_rows(76, n, Hkv * d).reshape(1, 1, n, Hkv * d)
            v = synth.normal_rows(77, n, Hkv * d).reshape(1, 1, n, Hkv * d)
            q = synth.normal(78, (n, H, d))
            _plant(what, at, k[0, 0], v[0, 0], q)
            c = Contig(backend, dtype, 1, 1, n, Hkv, d, k=k, v=v)
            for cap, window in ((None, None), (20.0, 37)):
                one = run_prefill(backend, c.cache, q, [0, n], [0], H, 0.1, cap, window)
                cuts = [0, 1, 30, 40, 41, 72, n]
                got = [run_prefill(backend, c.cache, q[a:b], [0, b - a], [a], H, 0.1, cap, window)
                       for a, b in zip(cuts, cuts[1:])]
                assert _same(np.concatenate(got), one), (what, at, cap, window)


@pytest.mark.parametrize("what", ["q_inf", "k_inf", "v_nan", "v_inf"])
@pytest.mark.parametrize("d,H,Hkv", [(64, 8, 2), (128, 8, 2), (256, 4, 2)])
def test_bf16_nonfinite_data_is_batch_invariant(backend, d, H, Hkv, what):
    """bf16 inputs: a prompt that starts inside a 32-key tile, with non-finite data beside its first rows, has the
    same bits alone (one 16-query tile per wave) as in a batch that fills the chip (two)."""
    n, off = 900 if d < 256 else 1700, 8
    k = synth.normal_rows(65, 8 * (n + off), Hkv * d).reshape(8, 1, n + off, Hkv * d)
    v = synth.normal_rows(66, 8 * (n + off), Hkv * d).reshape(8, 1, n + off, Hkv * d)
    q = synth.normal(67, (8 * n, H, d))
    for at in (40, 75, n - 20):
        k2, v2, q2 = k.copy(), v.copy(), q.copy()
        _plant(what, at, k2[0, 0], v2[0, 0], q2[:n])
        c = Contig(backend, "f32", 8, 1, n + off, Hkv, d, k=k2, v=v2)
        for window in (None, 50):
            both = run_prefill(backend, c.cache, q2, np.arange(9) * n, [off] * 8, H, 0.09, None, window, precision="bf16")
            alone = run_prefill(backend, c.cache, q2[:n], [0, n], [off], H, 0.09, None, window, precision="bf16",
                                seq_slot=np.array([0], np.int32))
            assert _same(alone, both[:n]), (what, at, window)


@pytest.mark.parametrize("d,H,Hkv,n", [(64, 4, 2, 90), (128, 4, 2, 200), (256, 4, 2, 90)])
def test_odd_values_reach_only_rows_that_attend_them(backend, d, H, Hkv, n):
    """Rows before a non-finite key or value have the bits of the clean prompt; rows from it on are non-finite in its
    own dimension alone (a value) or as 64 bits say (a key)."""
    at = n // 2 + 3
    k = synth.normal_rows(71, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    v = synth.normal_rows(72, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    q = synth.normal(73, (n, H, d))
    clean = run_prefill(backend, Contig(backend, "f32", 1, 1, n, Hkv, d, k=k, v=v).cache, q, [0, n], [0], H, 0.1)
    for what in ("v_nan", "v_inf", "k_inf", "v_max"):
        k2, v2, q2 = k.copy(), v.copy(), q.copy()
        _plant(what, at, k2[0, 0], v2[0, 0], q2)
        c = Contig(backend, "f32", 1, 1, n, Hkv, d, k=k2, v=v2)
        got = run_prefill(backend, c.cache, q2, [0, n], [0], H, 0.1)
        assert _same(got[:at], clean[:at]), what
        if what == "v_nan":
            bad = np.isnan(got[at:])
            assert bad[:, :H // Hkv, 7].all() and bad.sum() == (n - at) * (H // Hkv), what
        elif what == "v_inf":
            assert np.isposinf(got[at:, :H // Hkv, 7]).all() and np.isneginf(got[at + 3:, :H // Hkv, 9]).all()
        elif what == "v_max":
            assert np.isfinite(got).all()
            w = got[n - 1, 0, 3] / np.float64(3.4e38)  # the key's weight, all that counts in that dimension
            want = attention_f64(q[n - 1, 0], k[0, 0, :, :d], (np.arange(n) == at)[:, None] * np.ones(d), 0.1)[3]
            assert abs(w - want) <= 1e-5 * want
        else:  # a score is +inf (NaN row), or -inf: the key has no weight
            for r in range(at, n):
                if q[r, 0, 5] > 0:
                    kk, vv = np.delete(k[0, 0, :r + 1, :d], at, 0), np.delete(v[0, 0, :r + 1, :d], at, 0)
                    assert np.abs(got[r, 0] - attention_f64(q[r, 0], kk, vv, 0.1)).max() <= 1e-5
                else:
                    assert np.isnan(got[r, 0]).all()


@pytest.mark.parametrize("n", [9, 20, 31, 45])
@pytest.mark.parametrize("power", [-13, -16, -19, -25, -34])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_small_dimensions_keep_their_precision(backend, d, n, power):
    """V dimensions far below the others, in tiles that are not full and beside full ones: each against 64 bits,
    relative to its own largest value. The bound is that of the f32 sums: n products and n terms of the
    denominator, an ulp each, and the exponentials' few."""
    H, Hkv = 4, 2
    k = synth.normal_rows(81, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    v = synth.normal_rows(82, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    q = synth.normal(83, (n, H, d))
    v[..., 5::16] *= np.float32(2.0**power)
    c = Contig(backend, "f32", 1, 1, n, Hkv, d, k=k, v=v)
    got = run_prefill(backend, c.cache, q, [0, n], [0], H, 0.1)
    bound = (n + 8) * 2.0**-23
    for h in range(H):
        cols = slice(h // 2 * d, (h // 2 + 1) * d)
        kh, vh = k[0, 0, :, cols].astype(np.float64), v[0, 0, :, cols].astype(np.float64)
        for r in range(n):
            want = attention_f64(q[r, h], kh[:r + 1], vh[:r + 1], np.float64(np.float32(0.1)))
            err = np.abs(got[r, h] - want) / np.abs(vh[:r + 1]).max(0)
            assert err.max() <= bound, (h, r, int(err.argmax()), float(err.max()))


def _unit_scale():
    """The scale whose product with f32 log2(e) is 1, as the kernel forms it."""
    log2e = np.float32(1.4426950408889634)
    x = np.float32(np.log(2.0))
    for _ in range(8):
        if x * log2e == np.float32(1.0):
            return float(x)
        x = np.nextafter(x, np.float32(1.0) if x * log2e < 1 else np.float32(0.0), dtype=np.float32)
    raise AssertionError("no such scale")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("exponent", [20, 24, 25, 26, 27])
@pytest.mark.parametrize("tiles_apart", [True, False])
def test_scores_near_the_end_of_f32(backend, d, exponent, tiles_apart):
    """Scores of 2^20 to 2^27, whose ulps are an eighth to 16: the keys of each 32-key tile an ulp above the tile's
    before (tiles_apart), or scattered over 16 ulps. The scores and the differences that the softmax weighs are exact
    in f32; the result is finite and that of 64 bits."""
    H, Hkv, n = 4, 2, 150
    ulp = 2.0**(exponent - 23)
    k = np.zeros((1, 1, n, Hkv * d), np.float32)
    v = synth.normal_rows(91, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    q = np.zeros((n, H, d), np.float32)
    half = 2.0**(exponent // 2)
    q[:, :, 0] = half
    r = np.arange(n)
    step = r // 32 if tiles_apart else (r // 20 * 8 + r % 3) % 17  # in ulps of the score
    s = 2.0**exponent + step * ulp
    k[..., 0], k[..., d] = s / half, s / half
    assert (k[0, 0, :, 0].astype(np.float64) * half == s).all()
    c = Contig(backend, "f32", 1, 1, n, Hkv, d, k=k, v=v)
    got = run_prefill(backend, c.cache, q, [0, n], [0], H, _unit_scale())
    assert np.isfinite(got).all()
    for h in range(H):
        vh = v[0, 0, :, h // 2 * d:(h // 2 + 1) * d].astype(np.float64)
        for r in range(n):
            w = np.exp2(s[:r + 1] - s[:r + 1].max())
            want = w @ vh[:r + 1] / w.sum()
            assert np.abs(got[r, h] - want).max() <= 1e-5, (h, r)


@pytest.mark.parametrize("d,H,Hkv,seqs,cached", [(64, 8, 8, 16, 65000), (128, 8, 8, 5, 70000), (256, 4, 4, 3, 70000)])
def test_images_in_rounds_and_none(backend, d, H, Hkv, seqs, cached):
    """Contexts whose tile images pass the scratch bound several times: taken in rounds, and at d = 64 the last
    sequences past the last round convert their own tiles. Each has the bits of itself alone, and what it attends:
    every page of the table is one of a few physical pages, so 64 bits need the few."""
    page, pool_pages, rows = 16, 24, [35, 1, 20, 40]
    pool = backend.create_page_pool(pool_pages, Hkv, d, "f32")
    n = pool_pages * page
    k, v = synth.normal_rows(101, n, Hkv * d), synth.normal_rows(102, n, Hkv * d)
    pool.write_rows(np.arange(n, dtype=np.int64), k, v)
    lens = [rows[b % len(rows)] for b in range(seqs)]
    pages = (cached + max(lens) + page - 1) // page
    table = np.random.default_rng(103).integers(0, pool_pages, (seqs, pages)).astype(np.int32)
    q = synth.normal(104, (sum(lens), H, d))
    start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    both = run_prefill(backend, pool, q, start, [cached] * seqs, H, 0.1, table=table)
    for b in range(seqs):
        part = slice(start[b], start[b + 1])
        alone = run_prefill(backend, pool, q[part], [0, lens[b]], [cached], H, 0.1, table=table[b:b + 1])
        assert _same(alone, both[part]), b
        if b in (0, seqs - 1):  # the last row: each physical slot as often as the table names its page
            end = cached + lens[b]
            at = table[b, np.arange(end) // page].astype(np.int64) * page + np.arange(end) % page
            for h in (0, H - 1):
                cols = slice(h * Hkv // H * d, (h * Hkv // H + 1) * d)
                want = attention_f64(q[start[b + 1] - 1, h], k[at][:, cols], v[at][:, cols],
                                     np.float64(np.float32(0.1)))
                assert np.abs(both[start[b + 1] - 1, h] - want).max() <= 1e-5, (b, h)
    pool.destroy()
