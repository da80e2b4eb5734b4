"""The rANS encoder on the GPU divides the state by a frequency with one FP64
multiply-add (neuzip_amd/csrc/nz_kernels.hip, nz_quot and nz_quot_entry).  This
pins, in integer arithmetic on the host, that the low word of its result is the
exact quotient for every frequency, whatever cumulative frequency the multiplier's
low bits hold, and every state the encoder divides (16 <= x < f << 20)."""
import numpy as np


def _multiplier(f, low12):
    """bits of the table's double: (1 + 2^-39) / f times 2^1023, its last 12 bits replaced"""
    r = (np.float64(1.0) + np.float64(2.0 ** -39)) / np.float64(f)
    bits = int(r.view(np.uint64)) + (1023 << 52)
    return (bits & ~0xFFF) | low12


def test_low_word_is_the_quotient():
    for f in range(1, 4096):
        for low12 in (0, 4095):
            bits = _multiplier(f, low12)
            biased = bits >> 52
            assert 0 < biased < 2047  # finite, normal, positive
            mant = (bits & ((1 << 52) - 1)) | (1 << 52)
            # x is the subnormal x * 2^-1074, the multiplier is mant * 2^(biased - 1075); in units of
            # 2^-51 (the spacing of doubles in [2, 4)) their product is x * mant / 2^s and the addend
            # 2 - 2^-52 is 2^52 - 1/2
            s = 2098 - biased
            delta = f * mant - (1 << s)  # how far f * multiplier lies above 1
            # the one rounding gives floor(x / f) exactly if q < x * mant / 2^s < q + 1 for q = x // f.
            # Left side: smallest for x = q * f, where it reads q * delta > 0.
            assert delta > 0
            # Right side: largest for x = q * f + f - 1, where it reads (q + 1) * delta < mant.
            assert (1 << 20) * delta < mant
            # and the sum stays below 4, so that the spacing is the one assumed
            assert (((f << 20) - 1) * mant >> s) + (1 << 52) < 1 << 53


def test_bits_of_the_result_word():
    """The same with the roundings spelled out, on states at both ends of their quotients."""
    rng = np.random.default_rng(0)
    for f in (1, 2, 3, 5, 7, 64, 1000, 2049, 3001, 4094, 4095):
        low12 = int(rng.integers(0, 4096))
        bits = _multiplier(f, low12)
        mant, s = (bits & ((1 << 52) - 1)) | (1 << 52), 2098 - (bits >> 52)
        for q in [16, 17, 255, 4096, (1 << 20) - 2, (1 << 20) - 1] + [int(v) for v in rng.integers(16, 1 << 20, 50)]:
            for x in (q * f, q * f + f // 2, q * f + f - 1):
                num = 2 * x * mant + ((1 << 53) - 1 << s)  # twice the exact sum, over 2^s
                lo, rem = divmod(num, 2 << s)
                up = 2 * rem > (2 << s) or (2 * rem == (2 << s) and lo & 1)
                assert ((lo + up) & 0xFFFFFFFF) == q
