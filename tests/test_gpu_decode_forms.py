"""Both forms of the decode step: launches of up to 256 chunks read one prepared entry per step,
larger ones the slot table and the word in turn.  Chunk counts on both sides of the line, and
exponents that take words as slowly and as fast as a stream can.  Lossless, so the result is the
input bit for bit."""
import numpy as np
import pytest

from conftest import bf16_bits_normal
from test_gpu_parity import gpu_decode, gpu_encode

pytestmark = pytest.mark.gpu


def _bits(kind, n):
    rng = np.random.default_rng(n)
    low = rng.integers(0, 1 << 16, n, dtype=np.uint32) & 0x807F
    if kind == "normal":
        return bf16_bits_normal(n, seed=n & 0xFFFF)
    if kind == "constant":  # hardly a word in the whole record
        exps = np.full(n, 120)
    elif kind == "wide":  # close to 8 bits a symbol
        exps = rng.integers(0, 200, n)
    else:  # runs of rare symbols (12 bits each) in every lane at once, between runs that take nothing
        exps = np.full(n, 120)
        at = np.arange(n) // 4096 % 61 == 7
        exps[at] = rng.integers(0, 120, int(at.sum()))
    return (low | (exps.astype(np.uint32) << 7)).astype(np.uint16)


@pytest.mark.parametrize("kind", ["normal", "constant", "wide", "bursts"])
@pytest.mark.parametrize("chunk,lane,n", [(8192, 16, 256 * 8192), (8192, 16, 256 * 8192 + 1), (32768, 128, 600_011),
                                          (131072, 256, 1_000_003)])
def test_decode_forms(kind, chunk, lane, n):
    bits = _bits(kind, n)
    print(f"case {kind} chunk={chunk} lane={lane} n={n}", flush=True)
    comp, packed = gpu_encode(bits, 7, chunk, lane)
    rc, out = gpu_decode(comp, packed, n, 7, chunk, lane)
    assert rc == 0 and np.array_equal(out, bits)
