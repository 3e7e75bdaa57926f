"""GPU: batches whose shortest sequence must have more rows than the decode
classes take (num_tokens - (num_seqs - 1) * max_query_len tokens, at least)
launch no decode kernels.  A query tensor with rows past the last sequence
makes that bound too high: its short sequences then run as prefill."""
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, assert_close, batch_oracle, need_gpu, to_np_f32

DEV = "cuda"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens, extra, classes", [([90, 70, 100], 0, 0), ([40, 11], 0, 0), ([40, 10], 0, 2),
                                                    ([60, 2, 1], 120, 0)],
                         ids=["alike", "just_over", "just_under", "rows_past_the_end"])
def test_no_decode_classes(q_lens, extra, classes):
    need_gpu()
    announce(f"no decode classes {q_lens} +{extra}")
    b = W.build_batch([n + 200 for n in q_lens], q_lens, 48, 8, seed=sum(q_lens))
    T = b.num_tokens + extra
    info = gfx906_fa.plan_info(b.num_seqs, T, 48, 8, b.max_query_len, b.max_seq_len)
    assert info["decode_classes"] == classes  # 6 rows a token, 64 rows of decode tiles
    q = torch.zeros((T, 48, 128), dtype=b.query.dtype, device=DEV)
    q[:b.num_tokens] = b.query
    kp, vp = b.planes()
    out = gfx906_fa.paged_attention(q, kp, vp, b.block_table, b.seq_lens_t, b.qsl_t, b.max_query_len, b.max_seq_len,
                                    b.scale, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert_close(to_np_f32(out[:b.num_tokens]), batch_oracle(b))
