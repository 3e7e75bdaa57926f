"""GPU: the decode classes of mixed batches whose shortest sequence must have
more rows than they take (num_tokens - (num_seqs - 1) * max_query_len tokens,
at least): one class that takes every decode row count, since query rows past
the last sequence make that bound too high.  Where num_tokens itself shows
such rows, the classes are those of the batch without them."""
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, assert_close, batch_oracle, need_gpu, to_np_f32

DEV = "cuda"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens, heads, extra, classes", [
    ([90, 70, 100], (48, 8), 0, 1), ([40, 11], (48, 8), 0, 1), ([40, 10], (48, 8), 0, 2),
    ([60, 2, 1], (48, 8), 120, 2), ([100, 3, 1], (48, 8), 133, 1), ([512, 1], (64, 8), 15, 1),
    ([5] * 8, (6, 1), 8, 2), ([90, 1], (128, 1), 80, 0)],
    ids=["alike", "just_over", "just_under", "rows_past_the_end", "hidden_rows", "hidden_rows_64_8", "verify_padded",
         "no_class_holds_a_token"])
def test_decode_classes_with_rows_past_the_end(q_lens, heads, extra, classes):
    need_gpu()
    Hq, Hkv = heads
    announce(f"decode classes {q_lens} {heads} +{extra}")
    b = W.build_batch([n + 200 for n in q_lens], q_lens, Hq, Hkv, seed=sum(q_lens))
    T = b.num_tokens + extra
    info = gfx906_fa.plan_info(b.num_seqs, T, Hq, Hkv, b.max_query_len, b.max_seq_len)
    assert info["decode_classes"] == classes
    # every sequence of a decode row count (up to 64 rows) has a decode kernel
    G = Hq // Hkv
    assert all(n * G <= info["dec_rows_max"] for n in q_lens if n * G <= 64)
    q = torch.zeros((T, Hq, 128), dtype=b.query.dtype, device=DEV)
    q[:b.num_tokens] = b.query
    kp, vp = b.planes()
    out = gfx906_fa.paged_attention(q, kp, vp, b.block_table, b.seq_lens_t, b.qsl_t, b.max_query_len, b.max_seq_len,
                                    b.scale, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert_close(to_np_f32(out[:b.num_tokens]), batch_oracle(b))
