"""Rules of csrc/sh_gemm_plan.hpp that keep a product's precision, over the sizes models can have."""
import itertools

from plan import plans

# what dim, n_heads*head_dim and hidden can be
WIDTHS = (64, 128, 192, 256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096)
ROWS = (1, 4, 31, 64, 130, 255, 256, 257, 500, 1023, 1024, 1500, 4096)
COLS = sorted({*WIDTHS, *(2 * w for w in WIDTHS), 320, 2304, 16320, 16384, 32000, 50304})


def test_one_plane_where_it_has_always_been():
    """Long inputs and wide classifiers took one plane with K a multiple of 128 (each of their K
    ranges was one then), others from three K steps of 64 on; everything else kept the pair."""
    products = list(itertools.product(ROWS, COLS, WIDTHS, (1,)))
    for (m, n, k, _), p in zip(products, plans(products)):
        large = (m >= 1024 or (m >= 256 and n >= 16384)) and n % 128 == 0
        want = k % 128 == 0 if large else k // 64 >= 3
        assert p.one_plane_ok == want, (m, n, k)


def test_pairs_keep_sums_of_their_own():
    """A pair's lo products have a sum apart from the hi products' (k_gemm_ring's SEP) in all tiles but
    the widest, which only large products take."""
    products = [(m, n, k, 0) for m, n, k in itertools.product((*ROWS, 193, 700, 900), (*COLS, 6144, 2112), (*WIDTHS, 416, 1568))]
    for (m, n, k, _), p in zip(products, plans(products)):
        large = (m >= 1024 or (m >= 256 and n >= 16384)) and n % 128 == 0
        assert large or p.kind != "ring128x256", (m, n, k)
    # sizes that took them: two rounds of the next smaller tile
    assert {p.kind for p in plans([(193, 32000, 768, 0), (700, 6144, 2048, 0), (1000, 6144, 2048, 0)])} == {"ring128x128", "ring64x128"}


def test_sums_no_longer_than_those_of_the_ranges_before():
    """Large fp16 pairs of at most 384 tiles of 128 x 128, and others of K not a multiple of 64 and at most
    256 tiles of 64 x 64, were split into K ranges, each with one sum of 2 K / 32 / ranges products. Their
    sums have at most as many now: 16 steps of one plane, or all of a shorter K, then one addition per run."""
    products = [(m, n, k, 0) for m, n, k in
                itertools.product((*ROWS, 174, 300, 446), (*COLS, 2176, 3520, 6144), (*WIDTHS, 544, 1248, 1568, 1632, 2016, 2976))]
    seen = {True: 0, False: 0}
    for (m, n, k, _), p in zip(products, plans(products)):
        large = (m >= 1024 or (m >= 256 and n >= 16384)) and n % 128 == 0
        if p.few or (not large and k % 64 == 0):
            continue
        t = 128 if large else 64
        tiles = -(-m // t) * (n // t)
        ranges = max((r for r in (2, 3, 4) if k % (32 * r) == 0 and k // r >= 256 and tiles * r <= 768), default=1)
        if tiles >= 512 or ranges == 1:
            continue
        seen[large] += 1
        own = min(p.kc // 32, p.run or k)
        assert p.kind != "ring128x256" and own <= 2 * k // 32 // ranges, (m, n, k)
    assert min(seen.values()) > 50, seen
