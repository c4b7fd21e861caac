"""The decode that a shape is given to is the one that was measured faster there: us of the route taken / of the one it must not take."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat

# dtype, tokens, d_model, features, layers, survivors per source and token, tying, a top-k's list; route, us; other route, us
MEASURED = [
    ("float32", 522, 1024, 2960, 9, 18, "none", True, "thin", 167, "tiles", 278),
    ("float32", 199, 512, 1056, 15, 19, "none", True, "thin", 88, "tiles", 128),
    ("float32", 4907, 512, 2712, 4, 17, "none", True, "thin", 105, "gather", 184),
    ("float32", 777, 1024, 2216, 12, 16, "per_source", True, "thin", 326, "gather", 495),
    ("float32", 413, 2048, 8152, 4, 48, "none", False, "gather", 166, "tiles", 233),
    ("float32", 1186, 1024, 3232, 4, 38, "none", True, "gather", 120, "tiles", 157),
    ("float32", 1033, 2048, 1696, 13, 10, "per_source", False, "tiles", 985, "gather", 1713),
    ("float32", 7960, 256, 1648, 6, 9, "none", False, "tiles", 271, "gather", 401),
    ("float32", 1024, 768, 6144, 12, 200, "none", True, "tiles", 1469, "gather", 2618),
    ("bfloat16", 121, 1024, 4184, 15, 60, "none", True, "thin", 244, "tiles", 338),
    ("bfloat16", 374, 768, 2488, 10, 19, "none", True, "thin", 60, "tiles", 89),
    ("bfloat16", 936, 512, 4920, 9, 32, "none", True, "thin", 120, "gather", 200),
    ("bfloat16", 214, 1024, 2144, 10, 21, "none", True, "thin", 57, "gather", 96),
    ("bfloat16", 331, 1024, 13736, 11, 119, "none", True, "gather", 500, "tiles", 667),
    ("bfloat16", 573, 768, 5512, 15, 33, "per_source", False, "tiles", 278, "gather", 446),
    ("bfloat16", 3038, 512, 4608, 4, 24, "per_source", False, "tiles", 77, "gather", 111),
    ("bfloat16", 4096, 768, 24576, 12, 200, "none", True, "tiles", 2958, "gather", 6769),
]


@pytest.mark.parametrize("dtype,T,d,F,L,k,tying,selected,faster,us,slower,slower_us", MEASURED)
def test_the_faster_decode_is_taken(dtype, T, d, F, L, k, tying, selected, faster, us, slower, slower_us):
    assert us < slower_us
    lib = nat.load()
    args = (T, d, F, L, L, k * T * L, nat.TYING[tying], nat.dtype_code(getattr(torch, dtype)))
    tiles = lib.clt_decode_rows_wanted if dtype == "float32" else lib.clt_decode_tiles_wanted
    route = "thin" if selected and lib.clt_decode_thin_wanted(*args) else "tiles" if tiles(*args) else "gather"
    assert route == faster
