"""Which products of up to 16 rows leave the BLAS library for the weight-streaming kernel, how many rows of W its workgroups take, how many
tokens a strip of the norm with convolution, how many teams a workgroup of latent decode attention.  The sizes are those both sides were timed at, weights read from memory.  No GPU is needed."""
import ctypes
import os
import subprocess

import pytest

from polarquant_amd.modeling_common import _streams_faster

KERNEL = [(1, 16, 64), (8, 128, 4096), (16, 512, 4096), (8, 1024, 1024), (1, 4096, 4096), (16, 4096, 4096), (8, 3584, 3584), (1, 5120, 4096), (8, 6144, 4096),
          (8, 8192, 2048), (8, 14336, 4096), (4, 18944, 3584), (8, 32768, 2048), (1, 32768, 4096), (8, 128256, 4096), (8, 152064, 3584), (1, 4096, 14336),
          (8, 4096, 14336), (8, 3584, 18944), (8, 4096, 8192), (8, 8192, 8192), (4, 28672, 8192), (2, 8192, 28672), (8, 4096, 11008)]
LIBRARY = [(8, 128, 8192), (16, 128, 8192), (8, 256, 16384), (8, 512, 14336), (16, 512, 14336), (8, 1024, 8192), (12, 2048, 8192), (1, 16, 7168), (8, 64, 7168),
           (4, 5120, 5120), (8, 5120, 13824), (1, 4096, 16384), (1, 6144, 16384), (16, 6144, 4096), (12, 14336, 4096), (16, 32768, 4096), (9, 128256, 4096),
           (16, 152064, 3584), (9, 5120, 4096), (16, 4096, 14336), (9, 8192, 8192), (16, 8192, 4096), (12, 4608, 3584)]


@pytest.mark.parametrize("rows,n,k", KERNEL)
def test_the_kernel_takes(rows, n, k):
    assert _streams_faster(rows, n, k)


@pytest.mark.parametrize("rows,n,k", LIBRARY)
def test_the_library_keeps(rows, n, k):
    assert not _streams_faster(rows, n, k)


@pytest.fixture(scope="module")
def rules():
    here = os.path.dirname(os.path.abspath(__file__))
    os.makedirs(os.path.join(here, "_build"), exist_ok=True)
    so = os.path.join(here, "_build", "liblaunch_rules.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "c++", "-", "-o", so, "-I", os.path.join(os.path.dirname(here), "polarquant_amd", "csrc")],
                   input=b'#include "pq_linear_rules.h"\n#include "pq_steps_rules.h"\n#include "pq_latent_rules.h"\nextern "C" {\n'
                         b'int tiles(int m, int n, int ks, int mats) { return pq::small_m8_row_tiles(m, n, ks, mats); }\n'
                         b'int gelu_tiles(int m, int plain, int ff, int ks) { return pq::linear_gelu_row_tiles(m, plain, ff, ks); }\n'
                         b'int strip(int tokens, int taps, int pieces) { return pq::norm_conv_strip(tokens, taps, pieces); }\n'
                         b'int layout(int rank, int groups, int slices) { auto l = pq::latent_decode_layout(rank, groups, slices); return 1000 * l.teams + l.slices; }\n}', check=True)
    return ctypes.CDLL(so)


@pytest.fixture
def row_tiles(rules):
    return rules.tiles


@pytest.mark.parametrize("tokens,taps,pieces,want", [(8192, 4, 2, 32), (2048, 4, 2, 8), (512, 4, 2, 4), (6000, 4, 1, 16), (33, 4, 1, 4), (6000, 5, 1, 32), (6000, 8, 1, 32),
                                                     (6000, 12, 1, 32), (3000, 8, 1, 16), (700, 9, 2, 16), (300, 16, 2, 16), (300, 17, 2, 32), (3000, 9, 2, 32), (1500, 9, 2, 16),
                                                     (700, 9, 4, 32), (1500, 9, 4, 16), (700, 8, 4, 8)])
def test_strips_are_shortened_only_where_the_recomputed_norms_pay(rules, tokens, taps, pieces, want):
    assert rules.strip(tokens, taps, pieces) == want


@pytest.mark.parametrize("n,k,tiles", [(6144, 4096, [4] * 8), (10240, 4096, [2] * 8), (21504, 4096, [4] * 8), (4096, 4096, [2] * 8), (14336, 4096, [4] * 8),
                                       (28672, 4096, [2, 2, 2, 2]), (28672, 8192, [2, 2, 2, 2]), (43136, 4096, [2, 2, 2]), (8192, 8192, [2, 2, 2]), (5120, 13824, [2, 2])])
def test_tiles_of_the_faster_side(row_tiles, n, k, tiles):
    for rows, want in enumerate(tiles, 1):
        assert row_tiles(rows, n, 8 if k >= 8192 else 4, 1) == want, rows


def test_eight_tiles_only_where_x_is_what_costs(row_tiles):
    """32768 and 43136 outputs: 8 tiles gain 7 to 10 % with 8 rows and lose 4 to 5 % with one."""
    for n in (32768, 43136):
        assert row_tiles(8, n, 4, 1) == 8 and all(row_tiles(m, n, 4, 1) < 8 for m in (1, 2, 3, 4))


# rank, row tiles of all sequences, the plan's slices -> teams, slices
LATENT = [(512, 1, 96, 2, 96), (512, 8, 64, 2, 32), (512, 64, 8, 2, 4), (512, 86, 6, 2, 2), (512, 100, 6, 2, 2), (512, 129, 4, 2, 1), (512, 192, 3, 2, 1),
          (512, 256, 2, 2, 1), (512, 256, 1, 2, 1), (512, 257, 2, 1, 2), (512, 257, 1, 1, 1), (512, 300, 2, 1, 2), (512, 1024, 1, 1, 1),
          (256, 20, 5, 2, 5), (256, 20, 24, 2, 12), (256, 40, 13, 2, 6), (256, 64, 8, 2, 4), (256, 86, 6, 1, 6), (256, 129, 4, 1, 4), (256, 257, 2, 1, 2),
          (128, 20, 5, 2, 5), (128, 64, 5, 2, 4), (128, 65, 5, 1, 5), (128, 40, 13, 1, 13), (128, 86, 6, 1, 6), (128, 129, 4, 1, 4), (128, 300, 2, 1, 2),
          (64, 64, 8, 2, 8), (64, 64, 5, 2, 4), (64, 129, 4, 2, 4), (64, 300, 2, 2, 2), (64, 1024, 1, 2, 1)]


@pytest.mark.parametrize("rank,groups,slices,teams,used", LATENT)
def test_two_teams_only_where_a_round_of_workgroups_holds_them(rules, rank, groups, slices, teams, used):
    assert divmod(rules.layout(rank, groups, slices), 1000) == (teams, used)


def test_latent_plan_fills_the_units_with_workgroups_of_one_team():
    from polarquant_amd import _ffi
    plan = _ffi.latent_lib().pq_latent_decode_plan
    assert [plan(B, 1, 32, 1 << 20, 256) for B in (1, 8, 100, 129, 256, 257, 300, 512, 513)] == [512, 64, 6, 4, 2, 2, 2, 1, 1]
    assert [plan(8, 1, 32, keys, 256) for keys in (1, 128, 129, 1000)] == [1, 1, 2, 8] and plan(8, 1, 64, 1 << 20, 256) == 32


def test_tiles_around_a_shared_norm(row_tiles):
    """What the launches of the products around a norm rest on: two matrices with K split eight ways are never given four tiles, and one
    matrix no more than four up to the widest norm (8192)."""
    for rows in range(1, 9):
        assert all(row_tiles(rows, n, 8, 2) == 2 for n in range(16, 1 << 19, 16))
        assert all(row_tiles(rows, n, ks, 1) <= 4 for n in range(16, 8192 + 16, 16) for ks in (4, 8))
    assert next(n for n in range(16, 1 << 16, 16) if row_tiles(8, n, 4, 1) == 8) >= 28672


def test_cases_of_the_products_around_a_norm_select_their_launches(row_tiles):
    """The GPU tests' cases run each launch that there is: K split four and eight ways, two and four row tiles."""
    import test_shared_norm_gpu as t
    split = lambda k: 8 if k >= 8192 else 4
    gated = {(split(width), 2 if width >= 8192 else row_tiles(M, ff, 4, 2)) for M, width, ff in t.GATED_VARIANTS}
    into = {(split(k), min(4, row_tiles(M, width, split(k), 1))) for M, width, k in t.INTO_VARIANTS}
    assert gated == {(4, 2), (4, 4), (8, 2)} and into == {(4, 2), (4, 4), (8, 2), (8, 4)}


def test_cases_of_the_product_with_gelu_select_their_launches(rules):
    import test_recurrent_token_gpu as t
    older = [(8, 2, 8, 64, 40, 8192), (4, 4, 8, 18720, 14336, 4096), (4, 2, 5, 4096, 256, 2048), (1, 4, 6, 2048, 65536, 192), (1, 2, 1, 16, 8, 64)]
    seen = set()
    for ksplit, tiles, M, plain, ff, K in t.GELU_VARIANTS + older:
        ks = 8 if K >= 8192 else 4
        while ks > 1 and (K % (64 * ks) or K // (64 * ks) < 2):
            ks //= 2
        assert (ks, rules.gelu_tiles(M, plain, ff, ks)) == (ksplit, tiles)
        seen.add((ksplit, tiles))
    assert seen == {(ks, nt) for ks in (1, 2, 4, 8) for nt in (2, 4, 8)}
