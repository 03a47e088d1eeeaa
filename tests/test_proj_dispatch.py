"""Which kernel instances the projections' GPU tests reach (CPU only).

The rules of proj_gemm.hip and proj_lora.hip restated, with the tables and
limits read from the sources: every tile shape of both GEMMs, in both
directions, and every instance of lowrank_split has a case in
test_proj_fused_gpu.py, whatever the tables say later.
"""
import os
import re

import pytest

pytest.importorskip("torch")
import test_proj_fused_gpu as cases  # noqa: E402

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "glacier.tune_amd", "csrc")


def _source(name):
    with open(os.path.join(CSRC, name), encoding="utf-8") as f:
        return f.read()


GEMM, LORA = _source("proj_gemm.hip"), _source("proj_lora.hip")


def _up(a, b):
    return -(-a // b)


def _tiles(T, n_in, outs, backward, ft, tt):
    return (_up(n_in, ft) if backward else sum(_up(o, ft) for o in outs)) * _up(T, tt)


def _table():
    """(slots, us alone, us loaded, features, tokens) of kShapes."""
    rows = re.findall(r"^    GL_GEMM\((.*?)\),", GEMM, re.M)
    out = []
    for row in rows:
        slots, alone, loaded, _, fb, tb, wf, wt = [float(x.strip(" f")) for x in row.split(",")[:8]]
        out.append((int(slots), alone, loaded, int(32 * fb * wf), int(32 * tb * wt)))
    return out


def _dma_shape(T, n_in, outs, backward):
    def time(s):
        slots, alone, loaded, ft, tt = s
        full, rest = divmod(_tiles(T, n_in, outs, backward, ft, tt), slots)
        return full * loaded + (alone + (loaded - alone) * rest / slots if rest else 0.0)
    return min(_table(), key=time)


def _general_shape(bf16, T, n_in, outs, backward):
    big16, big32 = map(int, re.search(r"kBigTiles = sizeof\(IO\) == 2 \? (\d+) : (\d+);", GEMM).groups())
    if bf16 and min(n_in, *outs) < 8:
        return "tiny"
    return 128 if _tiles(T, n_in, outs, backward, 128, 128) >= (big16 if bf16 else big32) else 64


def _low_rank(T, jobs, rank, bf16, eights):
    tiles = _up(rank, 16)
    four, two = map(int, re.search(r"\(T \+ 63\) / 64 \* jobs >= (\d+)\) return 4;\s+"
                                   r"if \(\(T \+ 31\) / 32 \* jobs >= (\d+)\) return 2;", LORA).groups())
    cus = int(re.search(r"\(tiles \+ nt - 1\) / nt\) <= (\d+)\) return nt;", LORA)[1])
    if bf16 and eights and tiles <= 2 and _up(T, 64) * jobs >= four:
        return 4, tiles
    if _up(T, 32) * jobs >= two:
        return 2, tiles
    return 1, next((n for n in (1, 2) if _up(T, 16) * jobs * _up(tiles, n) <= cus), 4)


def _calls():
    """(bf16, T, in, outs, rank) of every case checked against float64."""
    bf16 = cases.torch.bfloat16
    yield from ((True, *c) for c in cases.SHAPES + cases.ODD_WIDTHS)
    yield from ((dtype == bf16, *c) for dtype, *c in cases.OTHER_SHAPES)
    for T, outs, rank in cases.RANKS:
        yield from ((dtype == bf16, T, n_in, outs, rank) for dtype, n_in in cases.RANK_WIDTHS)


def _eights(n_in, outs):
    return all(n % 8 == 0 for n in (n_in, *outs))


@pytest.mark.parametrize("backward", [False, True])
def test_every_tile_shape_has_a_case(backward):
    dma = {_dma_shape(T, n_in, outs, backward) for bf16, T, n_in, outs, _ in _calls()
           if bf16 and _eights(n_in, outs)}
    assert len(_table()) == 5
    assert dma == set(_table())
    general = {(bf16, _general_shape(bf16, T, n_in, outs, backward)) for bf16, T, n_in, outs, _ in _calls()
               if not (bf16 and _eights(n_in, outs))}
    assert general == {(True, "tiny"), (True, 64), (True, 128), (False, 64), (False, 128)}


def test_every_low_rank_instance_has_a_case():
    reached = set()
    for bf16, T, n_in, outs, rank in _calls():
        adapters = len(outs) - (len(outs) > 1)  # the second projection has none
        for jobs in (adapters, 2 * adapters):
            reached.add((bf16, _eights(n_in, outs), *_low_rank(T, jobs, rank, bf16, _eights(n_in, outs))))
    rows = {(1, 1), (1, 2), (1, 4), (2, 1), (2, 2), (2, 3), (2, 4)}
    assert {r[2:] for r in reached if not r[0]} == rows
    assert {r[2:] for r in reached if r[0] and not r[1]} == rows
    assert {r[2:] for r in reached if r[0] and r[1]} == rows | {(4, 1), (4, 2)}
