"""For which sizes the attention backward asks for scratch to keep dS in (a query that needs no GPU)."""
import ctypes as C

import pytest


@pytest.mark.parametrize("units,F,T,H,causal,kept", [
    # a pass of few or unevenly spread work-groups: the one grid of all passes is faster (26 against 31 us, 52 / 62, 33 / 29 ...)
    (86, 302, 77, 128, 0, False), (125, 276, 17, 192, 0, False), (87, 363, 77, 128, 0, False), (156, 182, 182, 192, 0, False),
    (269, 61, 61, 128, 1, False), (332, 49, 10, 80, 0, False), (81, 26, 443, 160, 0, False), (21, 277, 2006, 192, 0, False),
    (16, 2154, 2154, 160, 0, False), (24, 2048, 2048, 128, 1, False), (48, 54, 884, 72, 0, False), (16, 42, 3472, 256, 0, False),
    (255, 128, 128, 256, 0, False), (256, 2048, 2048, 64, 1, False),
    # enough of them: dS kept
    (256, 2048, 2048, 128, 1, True), (24, 2048, 2048, 128, 0, True), (32, 2048, 2048, 128, 1, True), (352, 180, 180, 128, 0, True),
    (352, 128, 128, 128, 0, True), (351, 128, 128, 128, 0, False), (261, 33, 65, 256, 0, True), (132, 129, 1, 200, 0, True),
    (16, 2048, 2048, 256, 1, True), (520, 1, 64, 72, 1, True), (196, 165, 38, 256, 0, True),
])
def test_scratch_that_keeps_score_gradients(xmk, units, F, T, H, causal, kept):
    L = xmk.lib()
    sizes = [C.c_uint32(x) for x in (1, units, H, F, T)]
    least, best = L.xmk_fmha_bwd_workspace_bytes(*sizes), L.xmk_fmha_bwd_best_workspace_bytes(*sizes, C.c_int32(causal))
    assert (best > least) == kept, (least, best)
