"""Query chunks of the global-row kernel (CPU; planning only). Grouped heads: at
least 256 queries a chunk over the heads of the kv group, no empty chunk. Packed
documents: cut only where the longest would outlast the others."""
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


@pytest.mark.parametrize("H,D,lens,chunks", [
    (32, 128, [2048] * 16, [1] * 16),        # two sweeps of 2002 queries a CU: even uncut
    (32, 128, [1024] * 16, [1] * 16),
    (16, 64, [4096] * 8, [4] * 8),           # 1.5 sweeps a CU: chunks of 1344
    (16, 64, [100] * 200, [1] * 200),
    (4, 128, [9001, 2048, 300], [47, 11, 2]),  # one long document: 417 a CU, chunks of 192
])
def test_document_chunk_counts(H, D, lens, chunks):
    W = [math.ceil(math.sqrt(n)) for n in lens]
    R = [n > 2048 for n in lens]
    rows = [-(-n // w) * (3 if r else 1) for n, w, r in zip(lens, W, R)]
    cu = [sum(lens[:i]) for i in range(len(lens) + 1)]
    p = N.problem(1, H, H, cu[-1], D, 0, any(R), 2, torch.float16, 0.1)
    need = N.workspace_bytes_varlen(p, N.Docs(cu, W, R))
    per_query = (H * cu[-1] * 4 + 255) // 256 * 256
    assert (need - 2 * per_query) // (H * 2 * D * 4) == sum(c * r for c, r in zip(chunks, rows))
