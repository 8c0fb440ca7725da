"""CPU: the density of the Lambertian (lisa_math.h) multiplies by the rounded
reciprocal of pi in 64 bits where the reference divides by pi: the same float for
every 24-bit significand.  Other exponents scale both sides exactly; where the
float result is denormal, its product with NdotL is zero either way."""
import numpy as np

PI = 3.14159265358979323846


def test_product_rounds_as_the_quotient():
    for first in range(0, 1 << 23, 1 << 21):
        x = (np.arange(first, first + (1 << 21), dtype=np.uint32) | np.uint32(0x3F000000)).view(np.float32)
        d = x.astype(np.float64)
        assert x[0] >= 0.5 and x[-1] < 1.0
        assert np.array_equal((d / PI).astype(np.float32), (d * (1.0 / PI)).astype(np.float32))


def test_denormal_densities_do_not_count():
    x = np.float32(2.0 ** -124)  # above it the quotient is a normal float
    for v in (x, np.float32(1e-40), np.float32(0.0)):
        for p in (np.float32(float(v) / PI), np.float32(float(v) * (1.0 / PI))):
            assert v * p == 0.0
