"""GPU: how a decode launch deals its sub-pages to workgroups: equal pieces of
each segment (aligned), or equal ranges over all segments with start-up units
in front of each (stream-K).  The published header says which ran; the pieces
it describes must cover every segment once, and the output, with and without
the folded cache write, must match the oracle."""
import numpy as np
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, assert_close, batch_oracle, need_gpu, to_np_f32

DEV = "cuda"
pytestmark = pytest.mark.gpu

rng = np.random.default_rng(3)
CASES = [
    # name, seq_lens, n_q, Hq, Hkv, aligned
    ("one_key", [1], 1, 48, 8, True),
    ("ragged_small", [900, 100, 33], 1, 48, 8, True),
    ("one_long", [12000], 1, 8, 1, True),
    ("even_fill", [2000] * 8, 1, 48, 8, True),
    ("ragged_ranges", rng.integers(200, 3000, 60).tolist(), 1, 48, 8, False),
    ("more_segments_than_workgroups", rng.integers(1, 400, 60).tolist(), 1, 48, 24, False),
    ("seventy_sequences", rng.integers(1, 900, 70).tolist(), 1, 8, 4, False),
    ("verify_ranges", rng.integers(60, 3000, 40).tolist(), 5, 48, 8, False),
    ("verify_even", [1500 + 5] * 4, 5, 6, 1, True),
    ("rows48", [5000, 700, 2500], 8, 6, 1, True),
    ("rows60_chunks", [300, 2000, 90], 10, 6, 1, True),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_decode_plan(case):
    need_gpu()
    name, lens, nq, Hq, Hkv, aligned = case
    announce(f"decode plan {name}")
    lens = [max(n, nq) for n in lens]
    b = W.build_batch(lens, [nq] * len(lens), Hq, Hkv, seed=sum(map(ord, name)))
    ws = gfx906_fa.new_workspace(gfx906_fa.workspace_size(b.num_seqs, b.num_tokens, Hq, Hkv, nq, max(lens)), DEV)
    out = W.attention(b, out_dtype=torch.float32, workspace=ws)
    torch.cuda.synchronize()
    U, nwg, upw, Uv, pad = ws[:40].view(torch.int64).cpu().tolist()
    pre = ws[256:256 + 4 * len(lens)].view(torch.int32).cpu().tolist()
    subs = [(n + 15) // 16 for n in lens]
    assert U == sum(subs) * Hkv and Uv == U + pad * len(lens) * Hkv and (upw > 0) == aligned, (U, nwg, upw, Uv, pad)
    if aligned:
        c = [-(-16 * n // upw) for n in subs]
        assert pre == [sum(c[:i]) for i in range(len(c))] and nwg == sum(c) * Hkv
    else:
        assert pre == [sum(subs[:i]) + pad * i for i in range(len(subs))]
    ref = batch_oracle(b)
    assert_close(to_np_f32(out), ref)
    # the last n_q tokens of each sequence written by the same launch
    at = np.cumsum(lens)
    new = torch.from_numpy(np.concatenate([np.arange(e - nq, e) for e in at])).to(DEV)
    kp, vp = b.planes()
    before = b.kv_cache.clone()
    for s in b.slot_mapping[new].tolist():  # wiped first: the call has to write them
        b.kv_cache[s // 16] = 0
    keep = torch.ones(len(b.slot_mapping), dtype=torch.bool, device=DEV)
    keep[new] = False
    gfx906_fa.reshape_and_cache_q8_kv(b.key[keep], b.value[keep], b.slot_mapping[keep], kp, vp)
    got = gfx906_fa.paged_attention(b.query, kp, vp, b.block_table, b.seq_lens_t, b.qsl_t, nq, max(lens), b.scale,
                                    out_dtype=torch.float32, workspace=ws, new_key=b.key[new], new_value=b.value[new],
                                    slot_mapping=b.slot_mapping[new])
    torch.cuda.synchronize()
    assert torch.equal(got, out) and torch.equal(b.kv_cache, before)
