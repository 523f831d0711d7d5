"""Attention of prompt portions over a bf16 cache at the edges of its kernel's blocks, against float64."""
import numpy as np
import pytest

import llama_box_amd as L
from test_gpu_nigozen import attention_case

pytestmark = pytest.mark.gpu


# cells: one block, a block and one cell, whole groups of four blocks and one more, many; queries: one wave, one more than two; long runs of hidden blocks in front (chunks)
@pytest.mark.parametrize("n_q,n_kv,heads,kv_heads,dk,dv,chunk,sink", [
    (32, 32, 2, 1, 128, 128, 0, True), (33, 33, 2, 2, 128, 128, 0, False), (65, 128, 4, 1, 128, 128, 64, True), (64, 161, 2, 1, 64, 64, 33, True),
    (130, 2100, 4, 2, 128, 128, 160, True), (40, 1500, 2, 1, 96, 96, 70, False), (100, 700, 2, 1, 128, 64, 0, True), (36, 260, 2, 1, 120, 96, 50, True), (300, 1030, 2, 1, 32, 32, 0, True)])
def test_prompt_attention_at_block_edges(backend, H, n_q, n_kv, heads, kv_heads, dk, dv, chunk, sink):
    """f32 sums of weights split into two bf16 terms (to 2^-17 of each): 2e-5 of the largest value"""
    rng = np.random.default_rng(n_q + 7 * n_kv)
    q = rng.standard_normal((n_q, heads, dk)).astype(np.float32)
    k = rng.standard_normal((n_kv, kv_heads, dk)).astype(np.float32)
    v = rng.standard_normal((n_kv, kv_heads, dv)).astype(np.float32)
    got, ref = attention_case(backend, H, L.BF16, n_q, n_kv, heads, kv_heads, dk, dv, chunk, sink, q, k, v, np.arange(n_kv - n_q, n_kv))
    assert np.abs(got - ref).max() <= 2e-5 * max(1.0, np.abs(ref).max())
