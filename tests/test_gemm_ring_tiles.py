"""Which kernel and tile a prompt's projection takes (host rules of
gemm_ring.hip and gemm_big.hip): a plain A never meets a tile that would
normalise it, and the MLP's output projection takes the faster kernel."""

import ctypes
import os

import pytest

from attention_nn_amd import _lib

STORE, RELU2, RESID_ATTN, RESID_MLP, LOGITS, QKV, CE = range(7)


@pytest.fixture(scope="module")
def tile():
    if not os.path.exists(_lib.LIB_PATH):
        from attention_nn_amd.build import build
        build()
    f = ctypes.CDLL(_lib.LIB_PATH)._ZN3ann14gemm_ring_tileEibiii
    f.argtypes, f.restype = [ctypes.c_int, ctypes.c_bool] + [ctypes.c_int] * 3, ctypes.c_int

    def call(epi, rms, M, N, K):
        t = f(epi, rms, M, N, K)
        return t >> 16, t & 0xffff
    return call


def _takes_rms(epi, bm, bn):
    """The small tiles of the qkv and fc epilogues form rms(A) in the product."""
    return epi in (STORE, RELU2, QKV) and bm * bn <= 128 * 64


@pytest.mark.parametrize("epi,cols", [(STORE, 3), (QKV, 3), (RELU2, 4), (RESID_ATTN, 1)])
def test_plain_product_never_takes_a_normalising_tile(tile, epi, cols):
    for d in (64, 128, 192, 512, 768, 1536):
        if epi == QKV and d % 128:
            continue
        for M in (129, 130, 300, 777, 1027, 2048, 4096, 8192, 32768):
            bm, bn = tile(epi, False, M, cols * d, d)
            assert bm and cols * d % bn == 0 and not _takes_rms(epi, bm, bn), (d, M, bm, bn)
            # the fastest tile of all where that one takes the rows as they are
            any_bm, any_bn = tile(epi, True, M, cols * d, d)
            assert _takes_rms(epi, any_bm, any_bn) or (any_bm, any_bn) == (bm, bn)


def test_columns_of_64_alone_have_no_plain_tile(tile):
    assert tile(STORE, False, 300, 320, 320) == (0, 0)
    assert tile(STORE, True, 300, 320, 320)[1] == 64
    assert tile(LOGITS, False, 300, 320, 320)[1] == 64


def test_gpu_cases_reach_every_tile(tile):
    """The row counts and widths of test_gpu_gemm_ring.py's cases, over the five
    products of a forward.  (A plain-store qkv has 3 d columns of an odd multiple
    of 64: never whole 128-column tiles.)"""
    from test_gpu_gemm_ring import CASES
    reached = set()
    for d, _, V, B, T in CASES:
        M, qkv = B * T, STORE if d % 128 else QKV
        shapes = [(qkv, True, 3 * d, d), (RELU2, True, 4 * d, d), (RESID_ATTN, False, d, d),
                  (RESID_MLP, False, d, 4 * d)] + ([(LOGITS, False, V, d)] if V % 64 == 0 else [])
        reached |= {(epi, tile(epi, rms, M, N, K)) for epi, rms, N, K in shapes}
    tiles = [(32, 64), (64, 64), (128, 64), (128, 128), (128, 192)]
    want = {(epi, t) for epi in (STORE, RELU2, RESID_ATTN, RESID_MLP, LOGITS) for t in tiles}
    want |= {(QKV, t) for t in [(64, 128), (128, 128), (192, 128)]}
    assert want - reached == {(STORE, (128, 128))}


# us behind the fc projection that writes A, on 256 CUs: the ring, the 256-row kernel
@pytest.mark.parametrize("d,M,ring,big", [
    (512, 16384, 35, 59), (512, 40960, 90, 122), (512, 65536, 167, 127), (512, 98304, 249, 195),
    (768, 8192, 52, 65), (768, 10240, 52, 66), (768, 19200, 108, 90), (768, 65536, 328, 298),
    (1024, 8192, 62, 104), (1024, 19200, 155, 213), (1024, 28000, 277, 231),
    (1024, 32768, 323, 261), (1024, 40960, 365, 324), (1280, 14000, 181, 237),
    (1280, 24576, 360, 301), (1280, 65536, 897, 718), (1536, 4096, 98, 121),
    (1536, 10240, 193, 164), (1536, 16384, 285, 261), (1536, 32768, 569, 512),
    (2048, 8192, 233, 213), (2048, 10240, 322, 374), (2048, 16384, 544, 472)])
def test_mlp_output_projection_takes_the_faster_kernel(tile, d, M, ring, big):
    f = ctypes.CDLL(_lib.LIB_PATH)._ZN3ann15gemm_big_routesEiii
    f.restype = ctypes.c_bool
    assert f(M, d, 4 * d) == (big < ring)
