"""The order in which the GEMM kernels' work-groups take the output tiles (csrc/tile_order.h), on the CPU, and what a work-group
waits for before it knows its tile, in the compiled kernels."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "intel-extension-for-openxla_amd", "csrc")

SOURCE = """
#include "tile_order.h"
using namespace gemm_impl;
extern "C" void tiles(uint32_t tiles_m, uint32_t tiles_n, int k, int slices, int* out) {
  const TileOrder o = slices ? tile_order_slices(tiles_m, tiles_n, k) : tile_order(tiles_m, tiles_n, k);
  for (uint32_t b = 0; b < tiles_m * tiles_n; ++b) {
    const TileAt t = tile_at(b, o);
    out[2 * b] = t.m;
    out[2 * b + 1] = t.n;
  }
}
extern "C" uint32_t quotient(uint32_t n, uint32_t d) { return tile_quotient(n, d, tile_inverse(d)); }
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_order")
    (d / "t.cc").write_text(SOURCE)
    so = str(d / "t.so")
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-D__forceinline__=inline", "-I", CSRC,
                           "-o", so, str(d / "t.cc")])
    L = C.CDLL(so)
    L.quotient.restype = C.c_uint32

    def tiles(tiles_m, tiles_n, k, slices):
        out = np.full((tiles_m * tiles_n, 2), -1, dtype=np.int32)
        L.tiles(C.c_uint32(tiles_m), C.c_uint32(tiles_n), C.c_int(k), C.c_int(slices), out.ctypes.data_as(C.c_void_p))
        return out
    return L, tiles


@pytest.mark.parametrize("k", [128, 129, 4096])
@pytest.mark.parametrize("slices", [0, 1])
def test_every_tile_once(order, slices, k):
    _, tiles = order
    grids = [(m, n) for m in range(1, 34) for n in range(1, 34)]
    grids += [(129, 2), (144, 2), (95, 3), (72, 4), (2, 129), (1, 4097), (4097, 1), (1023, 65), (257, 257), (8, 509)]
    for m, n in grids:
        t = tiles(m, n, k, slices)
        assert t.min() >= 0 and (t < [m, n]).all(), (m, n)
        assert len(np.unique(t[:, 0].astype(np.int64) * n + t[:, 1])) == m * n, (m, n)


def test_quotient_is_exact(order):
    L, _ = order
    top = 2 ** 32 - 1
    for d in (1, 2, 3, 5, 7, 8, 255, 4097, 65535, 65536, 1000003, 2 ** 31 - 1, 2 ** 31, 2 ** 31 + 1, top):
        for n in (0, 1, d - 1, d, d + 1, 2 * d - 1, 2 * d, top // d * d - 1, top // d * d, 2 ** 31, top - 1, top):
            if 0 <= n <= top:
                assert L.quotient(C.c_uint32(n), C.c_uint32(d)) == n // d, (n, d)


@pytest.mark.parametrize("header,kernel", [
    ("gemm_kernel.h", "gemm_mfma_kernel<_Float16, false, false, true, 64, 64, 2, 2, 64, 4>"),
    ("gemm_kernel.h", "gemm_mfma_kernel<__bf16, false, false, false, 128, 64, 2, 2, 64, 4>"),
    ("gemm_slices.h", "gemm_slices_kernel<_Float16, false, false, true, 1, 1, 4, false>"),
    ("gemm_ragged.h", "gemm_ragged_kernel<__bf16, false, false, true, 64, 2, true>"),
])
def test_first_loads_follow_one_round_of_arguments(tmp_path, header, kernel):
    """A launch of a few microseconds waits for its arguments once, not once for each use of them."""
    (tmp_path / "k.hip").write_text(f'#include "{header}"\ntemplate __global__ void gemm_impl::{kernel}(gemm_impl::GemmParams);\n')
    out = str(tmp_path / "k.s")
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                           "-Xclang", "-packed-fp32-ops", "--offload-device-only", "-S", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                           str(tmp_path / "k.hip"), "-o", out], stderr=subprocess.DEVNULL)
    lines = re.search(r"^_ZN9gemm_impl\S*:(.*?)s_endpgm", open(out).read(), re.M | re.S)[1].splitlines()
    first = next(i for i, l in enumerate(lines) if "buffer_load" in l or "global_load" in l)
    waits = [l for l in lines[:first] if "s_waitcnt" in l and "lgkmcnt" in l]
    assert len(waits) == 1 and not any("v_rcp" in l for l in lines[:first]), waits


@pytest.mark.parametrize("tiles_m,tiles_n", [(129, 2), (155, 2), (192, 2), (95, 3), (128, 3), (72, 4), (96, 4)])
def test_second_round_of_tall_outputs_rereads_rows(order, tiles_m, tiles_n):
    """A few tile columns and a long K, K split over the waves: what does not fit the first 256 work-groups takes rows of A that
    the first ones have read."""
    t = order[1](tiles_m, tiles_n, 4096, 1)
    assert set(t[256:, 0]) <= set(t[:256, 0])
