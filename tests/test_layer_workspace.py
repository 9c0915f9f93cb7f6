"""The layer workspace is no larger than Q8_K rows, two lists of 32-pair work
items and act rows of their own for the fused kernel took: a caller with a
buffer of a fixed size keeps the batches that fit it."""
import ctypes as C

import pytest

from zeromoe_amd._lib import ZmMoeLayer, ZmRouterSpec, lib

SYNC_BYTES = 4 * (16 * 33 + 2 * 1024 * 32)  # the fused kernel's counters


def _layer(H, F, E, K, NS, Fs):
    d = ZmMoeLayer()
    d.H, d.F, d.n_slots, d.router = H, F, NS, ZmRouterSpec(0, E, K, 0, 0, 0, 0.0)
    d.type_gate = d.type_up = d.type_down = 12
    d.w_gate = d.w_up = d.w_down = d.route_map = 256
    d.F_shared, d.type_shared = Fs, 12 if Fs else 0
    if Fs:
        d.ws_gate = d.ws_up = d.ws_down = 256
    return d


def _bytes(S, H, F, E, K, NS, Fs):
    def row(n):
        return (n // 256 * 292 + 15) // 16 * 16

    pairs = S * K
    items = ((pairs + 31) // 32 + min(pairs, NS)) * 4
    arrays = [S * E * 4, pairs * 4, pairs * 4, S * row(H), NS * 4, (NS + 1) * 4, pairs * 4, NS * 4, 4, items, 4, items,
              4, pairs * F * 4, pairs * row(F), pairs * H * 4]
    if Fs:
        arrays += [S * Fs * 4, S * row(Fs), S * H * 4]
    arrays += [(pairs * F + S * Fs) * 4]
    return sum((a + 255) // 256 * 256 for a in arrays) + SYNC_BYTES + 256


@pytest.mark.parametrize("Fs", [0, 256, 2048])
@pytest.mark.parametrize("H,F,E,K,NS", [(4096, 1536, 128, 8, 128), (7168, 2048, 256, 8, 96), (16384, 256, 8, 1, 8),
                                        (256, 256, 2, 2, 2), (2048, 768, 512, 10, 512)])
def test_no_larger_than_planar_rows_took(H, F, E, K, NS, Fs):
    L = lib()
    d = _layer(H, F, E, K, NS, Fs)
    for S in (1, 2, 8, 9, 33, 64, 333, 2048, 65535):
        assert 0 < L.zm_moe_workspace_size(C.byref(d), S) <= _bytes(S, H, F, E, K, NS, Fs), S
