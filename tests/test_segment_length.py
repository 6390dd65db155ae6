"""The automatic overlap-save segment length (dd_fdd_segment_length, host only)."""
import ctypes as C
import random

import pytest

FP32, BF16, FP16 = 0, 1, 2
VALU, TILE32, TILE16 = 0, 1, 2
LENGTHS = [8192, 16384, 32768, 65536, 131072, 262144]


@pytest.fixture
def segment_length(dd):
    fn = dd.lib().dd_fdd_segment_length
    fn.restype = C.c_size_t
    fn.argtypes = [C.c_int, C.c_int, C.c_size_t, C.POINTER(C.c_size_t), C.c_size_t, C.c_size_t, C.c_size_t]

    def call(form, prec, dmax, nsc, ndm, nchan):
        return fn(form, prec, dmax, (C.c_size_t * len(nsc))(*nsc), len(nsc), ndm, nchan)

    return call


@pytest.mark.parametrize("ndm", [1, 16, 20, 32, 64, 200, 256])
def test_few_trials_are_priced_as_a_whole_block(segment_length, ndm):
    """The contraction computes 256 DMs whatever the list holds: at 1024
    channels, 64701 samples and delays to 22527, 32768 takes 1.9 ms for 20 and
    for 256 trials, 65536 3.1 ms."""
    assert segment_length(TILE16, FP32, 22527, [64701 - 22527], ndm, 1024) == 32768


@pytest.mark.parametrize("form", [VALU, TILE32, TILE16])
@pytest.mark.parametrize("prec", [FP32, BF16, FP16])
def test_length_holds_the_largest_delay(segment_length, form, prec):
    for dmax in (0, 1, 8188, 8189, 65532, 65533, 262140):
        n = segment_length(form, prec, dmax, [1, 50000, 0], 700, 512)
        assert n in LENGTHS and n >= dmax + 4
    assert segment_length(form, prec, 262141, [1000], 700, 512) == 0


@pytest.mark.parametrize("nchan,nsc,ndm,dmax,want", [
    (64, [30770 - 3493] * 5, 78, 3493, 16384),     # 0.242 ms, 32768 0.294
    (1000, [252185 - 60000] * 5, 66, 60000, 131072),  # 17.5 ms, 262144 19.6
    (1024, [430837 - 12405], 373, 12405, 32768),   # 7.33 ms, 65536 7.81
])
def test_phasors_cost_what_the_tile_rule_says(segment_length, nchan, nsc, ndm, dmax, want):
    """Lengths that turn on the phasors' cost: priced as where the tiles of a
    chunk group are chosen, the faster of the two measured is taken."""
    assert segment_length(TILE16, FP32, dmax, nsc, ndm, nchan) == want


def _smallest_volume(dmax, nsc):
    """Chunk columns of the 16 x 16 tiles, padding included, times bins."""
    best = None
    for n in LENGTHS:
        if n < dmax + 4:
            continue
        good = (n - dmax) & ~1
        chunks = sum(-(-x // good) for x in nsc)
        groups, ntl = min(((-(-chunks // (8 * t)), t) for t in (1, 2, 3)),
                          key=lambda g: (g[0] * g[1] + 1.5 * g[0], -g[1]))
        cost = 8 * groups * ntl * (n // 2 + 1)
        if best is None or cost < best[0]:
            best = cost, n
    return best[1]


@pytest.mark.parametrize("prec", [BF16, FP16])
def test_reduced_precision_keeps_the_smallest_volume(segment_length, prec):
    """A segment with less padding holds a larger error in these forms: the
    estimated time, which takes such segments, is for float32 alone."""
    assert segment_length(TILE16, prec, 24849, [15625] * 8, 3000, 1024) == 65536
    assert segment_length(TILE16, FP32, 24849, [15625] * 8, 3000, 1024) == 32768
    rng = random.Random(7)
    for _ in range(400):
        dmax = rng.randint(0, 100000)
        nsc = [int(2 ** rng.uniform(10, 20)) for _ in range(rng.randint(1, 9))]
        assert segment_length(TILE16, prec, dmax, nsc, rng.randint(1, 3000), 1024) == _smallest_volume(dmax, nsc)
