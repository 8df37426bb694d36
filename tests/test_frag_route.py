"""The decode GEMM's choice of tile at the launches of a decode step, on each side of its lines (host
only: the choice reads sizes and pointer alignments)."""
import ctypes

import pytest

from vkwr_amd import capi

P = ctypes.c_void_p(0x100000)  # never dereferenced
RANKS = {768: (64, 64, 128, 64), 1024: (64, 64, 128, 32), 1536: (64, 64, 192, 64), 2048: (96, 96, 256, 64),
         2560: (96, 96, 320, 64), 3072: (96, 96, 384, 64), 4096: (128, 128, 480, 96)}


def problem(m, n, k):
    return capi.FragProblem(P, P, P, m, n, k, 0, 1, P, P, P)


def launch(kind, C, B):
    if kind == "out":
        return [problem(B, C, r) for r in RANKS[C]]
    if kind == "proj":
        return [problem(B, n, C) for n in (C, C, C, *RANKS[C])]
    return [problem(B, {"key": 4 * C, "o": C, "head": 65536}[kind], C)]


@pytest.mark.parametrize("kind,C,B,tile", [
    # low-rank outputs: up to 32 rows eight waves on 32 x 32, above small workgroups of four waves
    ("out", 4096, 1, (32, 32, 8)), ("out", 4096, 32, (32, 32, 8)), ("out", 2560, 16, (32, 32, 8)),
    ("out", 2048, 32, (32, 32, 8)), ("out", 4096, 33, (32, 64, 4)), ("out", 2048, 128, (32, 64, 4)),
    # K up to 1024: no more than two rounds (528 tiles) of 32 x 32
    ("proj", 768, 144, (32, 32, 8)), ("proj", 768, 192, (32, 32, 8)), ("proj", 768, 224, (64, 64, 8)),
    ("key", 768, 160, (32, 32, 8)), ("key", 768, 192, (64, 64, 8)), ("key", 1024, 128, (32, 32, 8)),
    ("proj", 1024, 129, (64, 64, 8)), ("key", 1024, 192, (64, 64, 8)),
    # one round of the smallest tile
    ("key", 2048, 32, (32, 32, 8)), ("key", 2048, 64, (32, 64, 8)), ("key", 2048, 128, (64, 64, 8)),
    ("key", 2048, 256, (128, 64, 4)), ("o", 2048, 160, (32, 64, 8)), ("key", 4096, 80, (128, 64, 4)),
    # beyond: four waves on 64 x 64 up to one and a half rounds of 128 x 64 or where those pad more rows
    ("proj", 2560, 256, (64, 64, 4)), ("key", 2560, 200, (64, 64, 4)), ("key", 3072, 256, (64, 64, 4)),
    ("proj", 4096, 256, (128, 64, 4)), ("key", 4096, 160, (64, 64, 4)), ("key", 4096, 256, (128, 64, 4)),
    ("head", 2048, 128, (128, 64, 4)), ("head", 2048, 32, (32, 64, 8)),
])
def test_tile_of_a_launch(kind, C, B, tile):
    assert capi.frag_route(launch(kind, C, B))[:3] == tile


@pytest.mark.parametrize("C,B,parts,tile", [
    (768, 64, 4, (32, 32, 8)), (768, 160, 3, (64, 64, 8)), (768, 224, 2, (32, 64, 8)), (2048, 32, 8, (32, 64, 8)),
    (2048, 128, 4, (64, 64, 8)), (2048, 160, 4, (128, 64, 4)), (2560, 160, 2, (64, 64, 8)),
])
def test_tile_of_a_k_split(C, B, parts, tile):
    assert capi.frag_route([problem(B, C, 4 * C)], parts)[:3] == tile
