"""Prompt portions whose keys are cut beside single tokens whose keys are cut: both kinds' parts are merged by one launch."""
import math

import pytest
import torch

from kernel_refs import PlainOps
from test_kernels_gpu import attention_tol, make_batch, make_paged_case

pytestmark = pytest.mark.gpu


# Single tokens in front of, between and behind the portions, of short and long contexts; three head sizes' merges; with a window; and so many single
# tokens that theirs come whole and only the portions' parts are left to merge.
@pytest.mark.parametrize("geometry,window,crowd", [((28, 4, 128, 16), None, 0), ((12, 2, 128, 32), 3000, 0), ((14, 2, 64, 16), None, 0),
                                                   ((28, 4, 128, 16), None, 300)])
def test_portions_and_single_tokens_merged_together(geometry, window, crowd):
    from tokenizer_amd.kernels import get_ops
    ops, ref = get_ops(), PlainOps()
    n_q, n_kv, d, page_size = geometry
    lengths, q_lens = [1700, 4220, 33, 340, 2500] + [20] * crowd, [1, 70, 1, 20, 1] + [1] * crowd
    qkv, k_pages, v_pages, positions, entry_of_token, table = make_paged_case(
        torch.bfloat16, n_q, n_kv, d, page_size, lengths=lengths, q_lens=q_lens, seed=31)
    parts = ops.lib.ta_prefill_attention_key_splits(sum(-(-n // 16) for n in q_lens if n > 1), n_q, n_kv, d, -1 if window is None else window,
                                                    ops.prefill_shape, max(lengths), ops.prefill_waves, ops.prefill_shared)
    assert parts > 1
    merged, real = [], ops.lib.ta_attention_merge_both
    out, want = torch.full((qkv.shape[0], n_q * d), float("nan"), dtype=torch.bfloat16).cuda(), torch.empty(qkv.shape[0], n_q * d, dtype=torch.bfloat16).cuda()
    scale = 1.0 / math.sqrt(d)
    ops.lib.ta_attention_merge_both = lambda *args: merged.append(1) or real(*args)
    try:
        ops.paged_attention(qkv, out, k_pages, v_pages, positions, entry_of_token, table, n_q, n_kv, d, window, scale,
                            max_position=max(lengths) - 1, batch=make_batch(lengths, q_lens))
    finally:
        ops.lib.ta_attention_merge_both = real
    ref.paged_attention(qkv, want, k_pages, v_pages, positions, entry_of_token, table, n_q, n_kv, d, window, scale)
    torch.testing.assert_close(out.float(), want.float(), **attention_tol(torch.bfloat16, True))
    assert len(merged) == (0 if crowd else 1)
