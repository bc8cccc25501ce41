"""How the weight gradient cuts an offset's pairs into chunks (host arithmetic, no GPU needed): longer chunks only where they
save a round of workgroups for less than they cost."""
import ctypes

import pytest

from warpconvnet_amd._lib import lib

STEP = 64
CHIP = 512  # workgroups of 128 x 128 channels that the chip holds


def _chunk(counts, c_in, c_out, identity=-1, identity_rows=0):
    offsets = [0]
    for n in counts:
        offsets.append(offsets[-1] + n)
    return lib().wcn_conv_wgrad_chunk_pairs((ctypes.c_int64 * len(offsets))(*offsets), len(counts), identity, identity_rows, c_in, c_out)


def _first(pairs, offsets, tiles):
    slots = CHIP // tiles
    want = max(64, slots // 2, slots - offsets // 2)
    return max(256, -(-(-(-pairs // want)) // STEP) * STEP)


def _most(counts, per):
    """Chunks of the XCD that has most of them."""
    here = [0] * 8
    for k, n in enumerate(counts):
        w = -(-n // per)
        starts = [0 if x * w <= (5 * k & 7) else (x * w - (5 * k & 7) + 7) // 8 for x in range(9)]
        for x in range(8):
            here[x] += starts[x + 1] - starts[x]
    return max(here)


@pytest.mark.parametrize("rows", [300, 24_000, 300_000])
@pytest.mark.parametrize("c_in,c_out,offsets", [(512, 640, 27), (512, 512, 125), (1024, 512, 27), (2048, 2048, 8), (4096, 4096, 27)])
def test_chunks_stay_as_they_are_where_longer_ones_would_not_fit_either(c_in, c_out, offsets, rows):
    tiles = (c_in // 128) * (c_out // 128)
    assert _most([rows] * offsets, 1 << 30) > CHIP // 8 // tiles  # one chunk each is too many
    assert _chunk([rows] * offsets, c_in, c_out) == _first(rows * offsets, offsets, tiles)


def test_chunks_stay_as_they_are_where_twice_their_length_would_not_fit_or_not_pay():
    for n in (24_000, 300_000):
        assert _chunk([n] * 27, 512, 512) == _first(27 * n, 27, 16)
    half = [2486, 6711, 2480, 7485, 11985, 7417, 2564, 6748, 2543, 6860, 11377, 6889, 12258]  # 24,000 rows of a room
    counts = half + [24_000] + half[::-1]
    first = _first(sum(counts) + 24_000, 27, 8)  # (the identity's rows and its pairs)
    assert _most(counts, first) > 8 >= _most(counts, 2 * first)  # 256 -> 512: two rounds of short chunks
    assert _chunk(counts, 256, 512, 13, 24_000) == first < _chunk(counts, 256, 256, 13, 24_000) * 2


@pytest.mark.parametrize("rows", [3_000, 24_000, 300_000])
@pytest.mark.parametrize("c_in,c_out", [(128, 128), (256, 256), (256, 512), (384, 384), (512, 128)])
def test_longer_chunks_fit_at_once_and_cost_less_than_the_rounds_they_save(c_in, c_out, rows):
    tiles, counts = (c_in // 128) * (c_out // 128), [rows // 5 + 37 * k for k in range(26)] + [rows]
    room, first, per = CHIP // 8 // tiles, _first(sum(counts), 27, tiles), _chunk(counts, c_in, c_out)
    rounds = -(-_most(counts, first) // room)
    assert per % STEP == 0 and first <= per
    if per > first:
        chunks = sum(-(-n // first) for n in counts)
        assert _most(counts, per) <= room < _most(counts, first) and per * chunks < rounds * sum(counts)


def test_what_lengthening_is_for():
    counts = [5_000 + 100 * k for k in range(26)] + [24_000]  # 256 -> 256: two rounds become one
    first = _first(sum(counts), 27, 4)
    assert _most(counts, first) > 16 and first < _chunk(counts, 256, 256) < 2 * first


def test_arguments_that_are_none():
    offsets = (ctypes.c_int64 * 3)(0, 10, 5)
    assert lib().wcn_conv_wgrad_chunk_pairs(offsets, 2, -1, 0, 64, 64) == 0
    assert lib().wcn_conv_wgrad_chunk_pairs(None, 2, -1, 0, 64, 64) == 0
    ok = (ctypes.c_int64 * 3)(0, 5, 10)
    assert lib().wcn_conv_wgrad_chunk_pairs(ok, 2, -1, 0, 60, 64) == 0
    assert lib().wcn_conv_wgrad_chunk_pairs(ok, 2, 1, 2**20, 64, 64) >= 256
