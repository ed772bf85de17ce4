"""The codebook decoder's group index (csrc/mq_codebook.hip, GroupIndex), restated: column k = 16 u of a weight
with groups of 16 d columns is in group u / d for every u < 2^26 and d < 2^26."""
import random

LIMIT = 1 << 26


def _constants(d):
    shift = max(d - 1, 0).bit_length()
    return -(-(1 << (26 + shift)) // d) << 5, shift


def test_equals_the_division():
    rng = random.Random(0)
    for d in [*range(1, 3000), *(1 << i for i in range(26)), *((1 << i) + 1 for i in range(1, 26)), LIMIT - 1,
              *(rng.randrange(1, LIMIT) for _ in range(3000))]:
        mul, shift = _constants(d)
        assert mul < 1 << 32
        top = (LIMIT - 1) // d
        for q in (0, 1, 2, top, rng.randint(0, top)):
            for u in (q * d - 1, q * d, q * d + 1, LIMIT - 1):
                if 0 <= u < LIMIT:
                    assert ((2 * u * mul) >> 32) >> shift == u // d
