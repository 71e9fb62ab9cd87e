"""Which kernel dense() takes (dih_dense_plan, no device needed)."""
import random

import pytest

import deepinfer_hip as dh
from tests import refcases

PLANE_BYTES = 32 << 20   # of one slot


def windows(columns):
    return columns // 256


@pytest.mark.parametrize("planes", [0, 1, 2])
def test_every_plan_can_be_launched(planes):
    """Over all the shapes that dense() takes: a width that is built, whole ranges with none
    empty, planes that fit their slot, no GEMM (and no bf16 weight copy) for short chunks."""
    rng = random.Random(planes)
    for _ in range(4000):
        rows = max(1, int(2 ** rng.uniform(0, 14.5)))
        columns = 64 * rng.randint(1, 128) if rng.random() < 0.3 else 512 * rng.randint(1, 16)
        tokens, bits = max(1, int(2 ** rng.uniform(0, 13.2))), rng.choice([5, 8])
        route, tiles, slabs, ranges = dh.dense_plan(rows, columns, bits, tokens, planes)
        may_gemm = tokens >= 1024 or (tokens >= 512 and rows <= 4096)
        at = (rows, columns, bits, tokens)
        if tokens <= 4:
            assert route == "gemv", at
        elif columns % 512:
            assert (route, tiles, slabs, ranges) == ("gemm" if may_gemm else "fused", 0, 1, 1), at
        elif route == "gemm":
            assert may_gemm, at
        elif tiles == 4:   # one round of blocks, one range
            assert (route, ranges) == ("fused", 1) and slabs in (1, 2), at
            assert -(-rows // (128 * slabs)) * -(-tokens // 128) <= 256, at
        else:
            assert route == "fused" and slabs == 1 and 1 <= tiles <= 3 and 1 <= ranges <= windows(columns), at
            per = -(-windows(columns) // ranges)
            assert per * (ranges - 1) < windows(columns), at
            if ranges > 1:
                items = -(-rows // 128) * -(-tokens // (32 * tiles))
                assert planes and ranges * items * 128 * 32 * tiles * 4 <= PLANE_BYTES, at


def test_refused_arguments():
    for args in [(0, 512, 8, 8), (512, 96, 8, 8), (512, 16384, 8, 8), (512, 512, 4, 8), (512, 512, 8, 0),
                 (512, 512, 8, 8, 3)]:
        with pytest.raises(dh.ArgumentError):
            dh.dense_plan(*args)


# Measured microseconds of a pass (one range, the best ranges): the second launch costs more than
# ranges give where K is short.
@pytest.mark.parametrize("bits,rows,columns,tokens,one,split", [
    (8, 512, 512, 16, 5.8, 9.0), (8, 2048, 512, 64, 5.6, 8.7), (8, 4100, 512, 33, 5.7, 8.7),
    (8, 8192, 512, 128, 6.5, 12.5), (8, 8192, 1024, 33, 8.7, 9.9), (8, 2048, 1024, 256, 8.9, 10.7),
    (8, 512, 1536, 16, 11.0, 9.3), (8, 512, 2048, 64, 14.0, 9.1), (8, 2048, 2048, 128, 14.2, 11.2),
    (8, 8192, 2048, 16, 14.0, 9.9)])
def test_ranges_where_they_pay(bits, rows, columns, tokens, one, split):
    assert (dh.dense_plan(rows, columns, bits, tokens)[3] > 1) == (split < one)


# Measured microseconds of a pass: blocks of 128 tokens and one or two 32-row slabs a wave fill the
# GPU in one round where the narrower blocks cross it.
@pytest.mark.parametrize("bits,rows,columns,tokens,slabs,narrow,wide", [
    (8, 8192, 2048, 896, 2, 54.6, 46.9), (8, 8192, 2048, 1000, 2, 55.0, 48.3), (5, 8192, 4096, 896, 2, 102.6, 88.5),
    (5, 16384, 2048, 512, 2, 58.2, 50.0), (8, 12288, 2048, 580, 2, 54.2, 47.3), (5, 12288, 2048, 640, 2, 57.9, 50.9),
    (5, 8192, 2048, 512, 1, 36.7, 33.0), (8, 8192, 4096, 512, 1, 54.8, 50.3), (5, 8192, 4096, 400, 1, 60.4, 54.6)])
def test_one_round_of_wide_blocks(bits, rows, columns, tokens, slabs, narrow, wide):
    assert dh.dense_plan(rows, columns, bits, tokens) == ("fused", 4, slabs, 1)


# Measured microseconds of a pass (fused, GEMM), with bf16 rows: past a thousand tokens a rule that
# ranks by launches of up to 1023 tokens took the fused kernel for all of these.
@pytest.mark.parametrize("bits,rows,columns,tokens,fused,gemm", [
    (8, 8192, 4096, 1800, 165.0, 135.4), (8, 4096, 4096, 3500, 163.2, 134.6), (8, 6001, 2048, 2100, 116.7, 95.8),
    (8, 12288, 2048, 3500, 234.0, 183.0), (8, 6001, 2048, 4096, 199.8, 159.4), (5, 6001, 2048, 4000, 200.1, 163.2),
    (8, 8200, 2048, 5000, 258.2, 183.1), (8, 8192, 2048, 5000, 226.8, 177.5), (8, 8200, 2048, 8192, 399.2, 287.3),
    # and where the fused kernel is the faster
    (8, 2048, 4096, 1280, 43.7, 61.2), (5, 4100, 512, 5000, 45.0, 86.5), (8, 8192, 2048, 1280, 69.5, 80.5),
    (8, 512, 2048, 640, 18.0, 22.4), (5, 4100, 512, 3000, 32.4, 51.9), (8, 4096, 2048, 1280, 38.8, 52.8)])
def test_long_chunks_take_the_faster_launch(bits, rows, columns, tokens, fused, gemm):
    assert dh.dense_plan(rows, columns, bits, tokens)[0] == ("gemm" if gemm < fused else "fused")


def test_fused_shapes_reach_every_form():
    """The GPU test's shapes run each width with one range, whole ranges and a shorter last one,
    and two slabs a wave, in both precisions."""
    forms = set()
    for bits in (8, 5):
        for rows, columns, tokens in refcases.DENSE_FUSED_SHAPES:
            route, tiles, slabs, ranges = dh.dense_plan(rows, columns, bits, tokens)
            assert route == "fused", (bits, rows, columns, tokens)
            short = windows(columns) % -(-windows(columns) // ranges) != 0
            forms.add((bits, tiles, "slabs" if slabs == 2 else "one" if ranges == 1 else "short" if short else "whole"))
    want = {(b, t, f) for b in (8, 5) for t in (1, 2, 3) for f in ("one", "whole", "short")}
    want |= {(b, 4, f) for b in (8, 5) for f in ("one", "slabs")}
    assert want - forms == set()


def gemm_block(rows, tokens):
    """The largest block whose tiles still give about one per CU."""
    for block in ((256, 256), (256, 128), (128, 128)):
        if -(-rows // block[0]) * -(-tokens // block[1]) >= 240:
            return block
    return 128, 64


@pytest.mark.parametrize("bits,rows,columns,tokens,y_bf16,block", refcases.DENSE_GEMM_SHAPES)
def test_gemm_shapes_reach_their_block(bits, rows, columns, tokens, y_bf16, block):
    assert dh.dense_plan(rows, columns, bits, tokens)[0] == "gemm" and gemm_block(rows, tokens) == block
    assert rows % block[0] != 0


def test_gemm_shapes_cover_every_block_and_store():
    got = {(block, rows * (2 if y_bf16 else 4) % 16 == 0)
           for _, rows, _, _, y_bf16, block in refcases.DENSE_GEMM_SHAPES}
    assert {b for b, _ in got} == {(256, 256), (256, 128), (128, 128), (128, 64)}
    assert {b for b, aligned in got if not aligned} == {(256, 256), (256, 128), (128, 128), (128, 64)}
