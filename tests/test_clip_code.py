"""The count pass's code of a clipped triangle (clip_code in
globalillumination_amd/csrc/raster_kernels.hpp), evaluated by the compiler: a
triangle past the clip list's capacity never reads as one within it, up to the
largest mesh's 2^28 - 1 clipped triangles, and no code names a tile."""
import subprocess

import pytest

from globalillumination_amd import build

SOURCE = """
#include "raster_kernels.hpp"
using namespace gi;
constexpr bool good(uint32_t c, uint32_t ccap) {
    const uint32_t code = clip_code(c, ccap);
    return (code & kClipCode) != 0 && ((code >> 18) & 15u) == 0 && clip_place(code) == (c < ccap ? c : ccap);
}
constexpr bool all(uint32_t ccap) {
    for (uint32_t c : {0u, 1u, 1023u, 16383u, 16384u, (1u << 18) - 1, 1u << 18, ccap - 1, ccap, ccap + 1,
                       (1u << 27) - 1, 1u << 27, (1u << 27) + 5, (1u << 28) - 1})
        if (!good(c, ccap)) return false;
    return true;
}
static_assert(all(CAPACITY), "clip_code");
"""


@pytest.mark.parametrize("capacity", ["wide_cap(0)", "kAttrTriangles", "wide_cap(5000000)", "wide_cap((1 << 28) - 1)"])
def test_places_past_the_list_stay_past_it(tmp_path, capacity):
    src = tmp_path / "clip_code.hip"
    src.write_text(SOURCE.replace("CAPACITY", capacity))
    cmd = [build._hipcc(), "-std=c++17", "--offload-arch=" + build.ARCH, "--cuda-host-only", "-fsyntax-only",
           f"-I{build.CSRC}", f"-I{build.ROOT / 'include'}", str(src)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
