"""Prefill's kernel variants: fp32 on split f16 pieces (staged and unstaged tiles, what the pieces cannot
carry, calls whose scratch cannot be had or whose tile images take several rounds), and one or two query
tiles per wave (both precisions)."""
from __future__ import annotations

import numpy as np
import pytest

from glint_amd import synth
from glint_amd.attn import GpuBackend
from gpu_util import Contig, run_prefill
from helpers import ABS_TOL, attention_f64

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("dtype", ["f32", "q8"])
@pytest.mark.parametrize("d,H,Hkv", [(64, 9, 3), (64, 8, 2), (128, 8, 2), (256, 4, 2)])
def test_staged_equals_unstaged(backend, dtype, d, H, Hkv):
    """A call of at most 96 rows per sequence converts tiles in its workgroups, a longer one stages them:
    a sequence has the same bits in either (rows on both sides of 16, 32 and 96)."""
    lens = [1, 15, 33, 95, 96, 97]
    offs = [40, 0, 70, 3, 31, 0]
    c = Contig(backend, dtype, len(lens), 1, 160, Hkv, d, seed=3100 + d + H)
    q = synth.normal(3200 + d, (sum(lens), H, d))
    start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    for cap, window in [(None, None), (20.0, 37)]:
        both = run_prefill(backend, c.cache, q, start, offs, H, 0.1, cap, window)
        few = len(lens) - 1
        alone = run_prefill(backend, c.cache, q[:start[few]], start[:few + 1], offs[:few], H, 0.1, cap, window)
        assert np.array_equal(_bits(alone), _bits(both[:start[few]])), (dtype, d, cap, window)


@pytest.mark.parametrize("precision", ["f32", "bf16"])
@pytest.mark.parametrize("d,H,Hkv,rows", [(64, 8, 2, 900), (128, 8, 2, 900), (256, 4, 2, 1700)])
def test_one_and_two_query_tiles_per_wave(backend, precision, d, H, Hkv, rows):
    """A call that fills the chip gives each wave two 16-query tiles, a smaller one (here the same prompts
    alone, a part-filled last tile included) one: the same bits."""
    lens = [rows, rows - 13, 200, rows, rows, rows, rows, rows]
    c = Contig(backend, "f32", len(lens), 1, rows, Hkv, d, seed=3300 + d)
    q = synth.normal(3400 + d, (sum(lens), H, d))
    start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    both = run_prefill(backend, c.cache, q, start, [0] * len(lens), H, 0.1, None, 333, precision=precision)
    for b in (0, 1, 2):
        part = slice(start[b], start[b + 1])
        alone = run_prefill(backend, c.cache, q[part], [0, lens[b]], [0], H, 0.1, None, 333, precision=precision,
                            seq_slot=np.array([b], np.int32))
        assert np.array_equal(_bits(alone), _bits(both[part])), (precision, d, b)


# (K row, V column, q row) multipliers of the values that leave the pieces' range, one at a time, and with
# how many keys: the bounds on K and V, and the spread inside a tile
@pytest.mark.parametrize("what", ["v_large", "v_small", "k_small", "q_small", "v_column", "k_row", "v_tiles", "zeros"])
@pytest.mark.parametrize("d,n", [(64, 40), (128, 131), (256, 40)])
def test_values_the_pieces_cannot_carry(backend, what, d, n):
    """Tiles and rows outside the pieces' range keep f32 precision: every output dimension against 64 bits,
    at the fp32 bar relative to that dimension's own V."""
    H, Hkv = 4, 2
    k = synth.normal_rows(41, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    v = synth.normal_rows(42, n, Hkv * d).reshape(1, 1, n, Hkv * d)
    q = synth.normal(43, (n, H, d))
    scale = 1 / np.sqrt(d)
    if what == "v_large":
        v *= np.float32(2.0**40)
    elif what == "v_small":
        v *= np.float32(2.0**-40)
    elif what == "k_small":
        k *= np.float32(2.0**-50)
        scale = 2.0**50 / np.sqrt(d)
    elif what == "q_small":
        q *= np.float32(2.0**-60)
        scale = 2.0**60 / np.sqrt(d)
    elif what == "v_column":
        v[..., 5::16] *= np.float32(2.0**-25)
    elif what == "k_row":
        k[:, :, 3::7] *= np.float32(2.0**-20)
    elif what == "v_tiles":  # tiles of different units, in range each
        v *= np.float32(2.0) ** (np.arange(n) // 32 * 9 % 30 - 15).astype(np.float32)[None, None, :, None]
    else:
        k[:, :, 32:], v[:, :, :32] = 0.0, 0.0
    c = Contig(backend, "f32", 1, 1, n, Hkv, d, k=k, v=v)
    got = run_prefill(backend, c.cache, q, [0, n], [0], H, scale)
    for h in range(H):
        cols = slice(h // 2 * d, (h // 2 + 1) * d)
        kh, vh = k[0, 0, :, cols].astype(np.float64), v[0, 0, :, cols].astype(np.float64)
        for r in range(n):
            want = attention_f64(q[r, h], kh[:r + 1], vh[:r + 1], scale)
            unit = np.abs(vh[:r + 1]).max(0) + 1e-300  # a dimension's own magnitude
            err = np.abs(got[r, h] - want) / unit
            assert err.max() <= ABS_TOL / 10, (what, h, r, int(err.argmax()), float(err.max()))


def test_capture_without_scratch():
    """fp32 prefill captured on a backend that has run nothing (no scratch to stage tiles in): accepted as
    before, and every replay gives the bits of the eager call."""
    be = GpuBackend(0)
    n, H, Hkv, d = 150, 8, 2, 128
    c = Contig(be, "f32", 1, 1, n, Hkv, d, seed=5)
    q = [synth.normal(6 + i, (n, H, d)) for i in range(3)]
    dq, dout = be.buffer(q[0]), be.empty(q[0].nbytes)
    qs, po = be.buffer(np.array([0, n], np.int32)), be.buffer(np.array([0], np.int32))
    graph = be.capture(lambda: be.prefill(c.cache, dq, dout, qs, po, 1, n, H, 0.09))
    got = []
    for x in q:
        dq.upload(x)
        graph.replay()
        be.sync()
        got.append(dout.download(x.shape))
    for x, y in zip(q, got):  # staged by now
        want = run_prefill(be, c.cache, x, [0, n], [0], H, 0.09)
        assert np.array_equal(_bits(y), _bits(want))
    graph.destroy()
    c.cache.destroy()
    be.close()


def test_tile_images_in_rounds(backend):
    """Storage so long that the images of all (sequence, KV head) pairs pass the scratch bound (16 pairs of
    64 MiB): the call runs in rounds, with the bits of each sequence alone."""
    H, Hkv, d, n, seqs, cap = 16, 8, 128, 100, 2, 65536
    cache = backend.create_kv_cache(1, cap, Hkv, d, "f32", seqs)
    offs = [70, 33]
    for b in range(seqs):
        rows = np.arange(offs[b] + n) + cache.row_id(b, 0, 0)
        cache.write_rows(rows, synth.normal_rows(50 + b, len(rows), Hkv * d), synth.normal_rows(60 + b, len(rows), Hkv * d))
    q = synth.normal(70, (seqs * n, H, d))
    both = run_prefill(backend, cache, q, [0, n, 2 * n], offs, H, 0.09)
    for b in range(seqs):
        alone = run_prefill(backend, cache, q[b * n:(b + 1) * n], [0, n], [offs[b]], H, 0.09,
                            seq_slot=np.array([b], np.int32))
        assert np.array_equal(_bits(alone), _bits(both[b * n:(b + 1) * n])), b
    cache.destroy()
