"""The polygon test's quotients: x times a double reciprocal, rounded to float, is the IEEE float quotient."""

import numpy


def test_product_with_double_reciprocal_is_the_float_quotient():
    """Random operands of every magnitude, and operands whose quotient lies next to a midpoint of floats."""
    rng = numpy.random.default_rng(3)
    n = 2000000
    f = numpy.float32

    def floats(k):
        return (rng.uniform(1, 2, k) * 2.0**rng.integers(-40, 40, k) * rng.choice([-1, 1], k)).astype(f)

    x, d = floats(n), floats(n)
    # x = d * (m + half an ulp of m) rounded up and down: quotients as near a midpoint as floats allow
    m = rng.uniform(1, 2, n).astype(f)
    near = d.astype(numpy.float64) * (m.astype(numpy.float64) + 2.0**-24)
    x = numpy.concatenate([x, near.astype(f), numpy.nextafter(near.astype(f), f(0)), f([0, -0.0, 1, numpy.inf])])
    d = numpy.concatenate([d, d, d, f([3, 3, numpy.inf, 2])])
    got = (x.astype(numpy.float64) * (1.0 / d.astype(numpy.float64))).astype(f)
    numpy.testing.assert_array_equal(got.view(numpy.uint32), (x / d).view(numpy.uint32))
    # a shorter reciprocal would not do
    assert ((x * (f(1) / d)).view(numpy.uint32) != (x / d).view(numpy.uint32)).any()
