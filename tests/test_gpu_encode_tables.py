"""Encode kernels against the oracle over the shapes of histogram that their
arithmetic depends on: frequencies from 1 to 4095, all 64 lanes of a wavefront
counting one symbol, an alphabet of everything, words in every step or in none;
for each segment-length class (8, 16, 32, 36 groups in registers, and longer)."""
import numpy as np
import pytest

from test_gpu_parity import gpu_decode, gpu_encode

pytestmark = pytest.mark.gpu


def _exponents(kind, n, rng):
    if kind == "constant":
        return np.full(n, 121, dtype=np.uint16)
    if kind == "two":  # one symbol in some fifty thousand: frequencies 4095 and 1
        return np.where(rng.random(n) < 2e-5, 3, 119).astype(np.uint16)
    if kind == "halves":  # each symbol halves the one before: frequencies 2048 down to 1
        return (127 - np.minimum(rng.geometric(0.5, n), 60)).astype(np.uint16)
    if kind == "everything":  # 256 symbols, most of them frequent enough to emit a word every other step
        return rng.integers(0, 256, n).astype(np.uint16)
    p = rng.dirichlet(np.full(40, 0.3))  # uneven
    return (90 + rng.choice(40, size=n, p=p)).astype(np.uint16)


@pytest.mark.parametrize("chunk,lane", [(32768, 64), (65536, 128), (65536, 256), (131072, 256), (147456, 288), (196608, 384)])
@pytest.mark.parametrize("kind", ["constant", "two", "halves", "everything", "uneven"])
def test_histogram_shapes(oracle, kind, chunk, lane):
    rng = np.random.default_rng(chunk + lane)
    n = 2 * chunk + 64 * lane + 777  # two whole chunks, one whole segment of a third, a ragged group
    bits = rng.integers(0, 1 << 16, n).astype(np.uint16) & 0x807F | (_exponents(kind, n, rng) << 7)
    print(f"case {kind} chunk={chunk} lane={lane}", flush=True)
    comp, packed = gpu_encode(bits, 7, chunk, lane)
    o_comp, o_packed = oracle.compress_bf16(bits, 7, chunk, lane)
    assert np.array_equal(packed.cpu().numpy(), o_packed)
    assert np.array_equal(comp.cpu().numpy(), o_comp)
    rc, out = gpu_decode(comp, packed, n, 7, chunk, lane)
    assert rc == 0 and np.array_equal(out, bits)
