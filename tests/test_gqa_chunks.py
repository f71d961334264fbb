"""Query chunks of the global-row kernel with grouped heads (CPU; planning only):
at least 256 queries a chunk over the heads of the kv group, no empty chunk."""
import ctypes
import math

import pytest
import torch

from cron_root_attention import _native as N


@pytest.mark.parametrize("B,Hq,Hkv,S,D,chunks", [
    (2, 16, 2, 2048, 64, 32),    # 64 queries a chunk, the least
    (1, 8, 1, 4096, 128, 64),
    (1, 32, 8, 2000, 128, 32),   # 63 queries of four heads, rounded to 64
    (1, 4, 2, 300, 64, 3),       # 300 * 2 / 256, rounded up: 100 queries, rounded to 128
    (1, 16, 4, 16000, 128, 42),  # 1.5 rounds of the CUs: 48 chunks of 384, 42 not empty
    (1, 16, 16, 16000, 128, 12),
])
def test_chunk_counts(B, Hq, Hkv, S, D, chunks):
    lib = N.load_library()
    relay = S > 2048
    p = N.problem(B, Hq, Hkv, S, D, math.ceil(math.sqrt(S)), relay, 2, torch.float16, 0.1)
    need = lib.cra_bwd_workspace_bytes(ctypes.byref(p))
    per_query = (B * Hq * S * 4 + 255) // 256 * 256
    per_chunk = B * Hkv * lib.cra_global_rows(ctypes.byref(p)) * 2 * D * 4
    assert (need - 2 * per_query) % per_chunk == 0
    assert (need - 2 * per_query) // per_chunk == chunks
