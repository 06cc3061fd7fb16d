"""The rule by which the prefill GEMM takes a kernel form (q27x_gemm_i8g_form), on the host: every form it may choose
fits the shape, none is listed in vain, and shapes of many short blocks or of small groups get tiles that suit them."""
import ctypes
import random

import pytest

# the launcher's lists: (tokens, weight rows) of a tile
FORMS_K = [(16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (64, 256), (128, 128), (128, 256), (256, 128), (256, 256),
           (128, 128), (256, 128), (256, 128)]
FORMS_G = [(16, 32), (32, 32), (32, 64), (64, 128), (64, 256), (128, 128), (128, 256), (256, 128), (256, 128), (128, 128),
           (256, 128)]


def form(X, M, N, K, gs):
    bm, bn = ctypes.c_int(), ctypes.c_int()
    i = X.lib().q27x_gemm_i8g_form(M, N, K, gs, ctypes.byref(bm), ctypes.byref(bn))
    return i, (bm.value, bn.value)


@pytest.fixture(autouse=True)
def plain_rule(monkeypatch):
    monkeypatch.delenv("Q27X_GEMM_FORM", raising=False)
    monkeypatch.delenv("Q27X_GEMM_W4", raising=False)


def test_forms_fit_and_all_are_used(X):
    """Over the shapes that callers bring, with whole 128-byte stages and below 2 GiB of codes: the form's tile divides N
    and is the list's, and every form is chosen, but the last three of the first list (shapes that nothing else takes)."""
    seen = {True: set(), False: set()}
    for N in (128, 256, 640, 1024, 2048, 4096, 5120, 10240, 14336, 16384, 34816, 62080):
        for K in (128, 256, 512, 1024, 1408, 2048, 3200, 4096, 5120, 6144, 17408):
            for M in (1, 9, 16, 30, 48, 64, 100, 128, 203, 256, 384, 511, 512, 700, 1024, 1536, 2048, 3000, 4096):
                for gs in [K] + [g for g in (128, 256, 512, 640, 1024) if K % g == 0 and 1 < K // g <= 20]:
                    i, tile = form(X, M, N, K, gs)
                    forms = FORMS_K if gs == K else FORMS_G
                    assert 0 <= i < len(forms) and tile == forms[i] and N % tile[1] == 0, (M, N, K, gs, i, tile)
                    if tile == (256, 256) or (gs != K and i == 8):
                        assert M >= 512 and K % 256 == 0 if gs != K else M >= 512, (M, N, K, gs)
                    if gs != K and tile[0] + tile[1] >= 384 and i in (6, 7):
                        assert K // gs <= 10, (M, N, K, gs)
                    seen[gs == K].add(i)
    assert seen[True] == set(range(10)) and seen[False] == set(range(11)), seen


@pytest.mark.parametrize("M,N,K,gs,least", [
    (33, 36864, 512, 512, 64 * 128),         # few K stages, many weight rows: 21 us in 32 x 64 split-K tiles, 10 in larger ones
    (48, 36864, 512, 512, 64 * 128), (47, 36864, 512, 512, 64 * 128),
    (16, 36864, 512, 256, 64 * 128),         # the same in groups
    (64, 19328, 1408, 1408, 64 * 128),
    (512, 4096, 256, 128, 64 * 128),         # groups of one stage: 25 us in 32 x 32 tiles, 9
    (384, 14336, 5120, 256, 128 * 128),      # 20 folds per tile: 93 us in 64 x 128 tiles, 70 in 128 x 128
    (1, 62080, 5120, 256, 128 * 128),        # 104 us in 64 x 128, 82 in 128 x 128
])
def test_short_blocks_and_small_groups_take_larger_tiles(X, M, N, K, gs, least):
    i, (bm, bn) = form(X, M, N, K, gs)
    assert bm * bn >= least, (i, bm, bn)


def test_small_m_keeps_the_split_k_tiles(X):
    for N, K in ((5120, 17408), (5120, 6144), (16384, 5120), (10240, 5120)):
        for M in (1, 8, 16):
            assert form(X, M, N, K, K)[1] == (16, 32)
            if K % 1024 == 0:
                assert form(X, M, N, K, 1024)[1] == (16, 32)


def test_general_forms_take_the_rest(X):
    for gs in (1088, 64):                                        # half a 128-byte stage left over
        for M, tile in ((1, (128, 128)), (511, (128, 128)), (512, (256, 128)), (4096, (256, 128))):
            assert form(X, M, 256, 1088, gs)[1] == tile
    assert form(X, 600, 128, 1280, 320)[1] == (256, 128)         # groups of half stages
    # 2 GiB of codes and more: 64-bit addresses
    assert form(X, 600, 1 << 18, 8192, 8192) == (12, (256, 128))
    assert form(X, 600, 1 << 18, 8192, 1024)[0] == 8
    assert form(X, 100, 1 << 18, 8192, 8192) == (10, (128, 128))
    for bad in ((1, 100, 1024, 1024), (1, 128, 1000, 1000), (1, 128, 2048, 192), (1, 128, 43008, 1024), (0, 128, 128, 128),
                (1, 128, 128, 0)):
        assert X.lib().q27x_gemm_i8g_form(*bad, None, None) == -2, bad


def test_drawn_shapes_have_a_form(X):
    rng = random.Random(3)
    for _ in range(3000):
        K = 64 * rng.randint(1, 300)
        gs = K // rng.choice([d for d in range(1, 21) if K % d == 0 and (K // d) % 64 == 0])
        N, M = 128 * rng.randint(1, 300), rng.randint(1, 4096)
        i, (bm, bn) = form(X, M, N, K, gs)
        assert i >= 0 and N % bn == 0
        if K % 128 or gs % 128:
            assert (bm, bn) == ((128, 128) if M < 512 else (256, 128))
