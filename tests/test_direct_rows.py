"""cra_reads_global_rows: which calls need packed global rows, and what the
in-place entry points refuse (CPU; nothing is launched and no pointer is read)."""
import ctypes
import math

import pytest
import torch

from cron_root_attention import _native as N


def reads(S, relay, ss, dtype=torch.float16, W=None, vss=None):
    p = N.problem(1, 2, 2, S, 64, W or max(1, math.ceil(math.sqrt(S))), relay, 2, dtype, 0.125)
    t = N.CraTensor(0x10000, 2 * S * ss, S * ss, ss)
    u = N.CraTensor(0x10000, 2 * S * (vss or ss), S * (vss or ss), vss or ss)
    return N.load_library().cra_reads_global_rows(ctypes.byref(p), t, u)


@pytest.mark.parametrize("S,relay,ss,want", [
    (1, False, 64, 0),
    (2048, False, 64, 0),
    (2048, False, 32 * 64, 0),
    (100000, False, 64, 0),     # no relay by choice
    (2048, True, 64, 1),        # relay rows are packed
    # strides whose tiles, 64 rows of W past the last row, would wrap 32 bits
    (2, False, 1 << 24, 1),     # (2 + 64 * 2) * 2^25
    (62, False, 1 << 22, 1),    # (62 + 64 * 8) * 2^23 > 2^32
    (62, False, 1 << 21, 0),    # half of that
])
def test_which_calls_read_packed_rows(S, relay, ss, want):
    assert reads(S, relay, ss) == want


def test_k_and_v_of_different_strides():
    assert reads(100, False, 64, vss=128) == 1


def test_wider_elements_halve_the_limit():
    assert reads(62, False, 1 << 21, torch.float32) == 1


def test_invalid_problem():
    assert reads(10, False, 64, W=11) == -1


@pytest.mark.parametrize("relay,vss,hkv,code", [
    (1, 64, 2, N.E_LAYOUT),        # relay rows are packed
    (0, 128, 2, N.E_LAYOUT),       # k and v of different row strides
    (0, 64, 65536, N.E_INVALID),   # the limit of cra_build_global
])
def test_inplace_refuses(relay, vss, hkv, code):
    lib = N.load_library()
    p = ctypes.byref(N.problem(1, hkv, hkv, 100, 64, 10, relay, 2, torch.float16, 0.125))
    t, v = N.CraTensor(0x10000, 6400 * hkv, 6400, 64), N.CraTensor(0x10000, 100 * vss * hkv, 100 * vss, vss)
    assert lib.cra_fwd_inplace(p, t, t, v, t, 0x10000, None) == code
    assert lib.cra_bwd_inplace(p, t, t, v, t, t, 0x10000, t, t, t, 0x10000, 1 << 40, None) == code
