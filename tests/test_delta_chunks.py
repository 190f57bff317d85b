"""What the chunked delta rule's entry point refuses, without a GPU: a step of no tokens launches nothing."""

import ctypes

import pytest

from halite_amd.kernels import library


def call(places, w_dtype=0, dtype=0, D=64, rate=0.6):
    """The entry point's answer for a step of no tokens; ``places``: how many bytes past a multiple of 16 arguments lie."""
    lib = library.core_library()
    at = lambda name: ctypes.c_void_p((1 << 20) + places.get(name, 0))  # noqa: E731
    n = 4 * D
    return lib.hal_delta_chunks(
        at("r"), n, at("k"), n, at("v"), n, at("a"), n, at("x1"), 8, at("w2"), at("w0"), at("a_bias"), w_dtype, 8, ctypes.c_float(rate),
        ctypes.c_float(1e-6), at("records"), at("state"), at("starts"), at("lens"), at("slots"), at("z"), n, at("weight"), w_dtype,
        ctypes.c_float(1e-5), at("out"), dtype, 0, 0, 4, D, ctypes.c_void_p(0))


@pytest.mark.parametrize("dtype", [0, 1])
def test_places(dtype):
    assert call({}, dtype=dtype) == 0
    assert call(dict(w2=4, w0=2, a_bias=2, weight=2, r=4, k=4, a=4, x1=4), w_dtype=1, dtype=dtype) == 0  # (read one by one there)
    assert call(dict(records=8), dtype=dtype) != 0 and call(dict(out=4), dtype=dtype) != 0
    assert call(dict(v=8), dtype=dtype) != 0 and call(dict(z=4), dtype=dtype) != 0
    assert (call(dict(out=8), dtype=dtype) == 0) == (dtype == 1)


def test_sizes():
    assert call({}, D=128) != 0 and call({}, rate=2.6) != 0
