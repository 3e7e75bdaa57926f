"""GPU: the one-wave prefill plan (at most 64 sequences and 64 row tiles).
The work list it leaves in the workspace must hold every (sequence, row tile)
once, whole or as pieces that cover its key tiles in order, with the
sequence's scalars, distinct partial slots that the split list names, and the
longest items first where they take more than one round of workgroups."""
import numpy as np
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, assert_close, batch_oracle, need_gpu, to_np_f32

DEV = "cuda"
pytestmark = pytest.mark.gpu

CASES = [
    # name, seq_lens, q_lens, Hq, Hkv
    ("one_tile", [900], [43], 48, 8),
    ("one_tile_6_1_long", [20000], [100], 6, 1),                # one row tile cut for 256 workgroups
    ("rows128_x8", [5000 + 7 * i for i in range(8)], [12] * 8, 48, 8),
    ("ragged_decode_between", [300, 1, 700, 40, 1200], [300, 1, 0, 40, 1200], 48, 8),
    ("sixty_three_tiles", [2016], [2016], 8, 1),
    ("two_rounds_uneven", [64 * (i % 9 + 1) + 40 for i in range(30)], [40] * 30, 48, 8),
    ("two_rounds_even", [2000] * 33, [33] * 33, 48, 8),
    ("more_than_two_rounds", [1500 + 100 * i for i in range(20)], [70] * 20, 32, 32),
    ("sixty_sequences", [70 + i for i in range(60)], [1] * 59 + [70], 6, 1),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_wave_plan(case):
    need_gpu()
    name, sls, qls, Hq, Hkv = case
    announce(f"wave plan {name}")
    b = W.build_batch(sls, qls, Hq, Hkv, seed=sum(map(ord, name)))
    info = gfx906_fa.plan_info(b.num_seqs, b.num_tokens, Hq, Hkv, b.max_query_len, b.max_seq_len)
    assert info["pf_items_max"] <= 64 and b.num_seqs <= 64  # the one-wave kernel
    ws = gfx906_fa.new_workspace(info["img_offset"], DEV)
    out = W.attention(b, out_dtype=torch.float32, workspace=ws)
    torch.cuda.synchronize()
    off, cap = info["pf_header_offset"], info["pf_grid_items"]
    total, nsplit = ws[off:off + 8].view(torch.int32).cpu().tolist()
    assert 0 < total <= cap
    items = ws[off + 256:off + 256 + 48 * total].view(torch.int32).view(total, 12).cpu().numpy()
    so = off + 256 + (48 * cap + 255) // 256 * 256
    split = {(e[0], e[1]): (e[2], e[3]) for e in ws[so:so + 16 * nsplit].view(torch.int32).view(-1, 4).cpu().tolist()}
    assert len(split) == nsplit
    G, R, qsl = Hq // Hkv, info["pf_rows"], b.qsl
    ntk, rows = {}, {}
    for s, (sl, nq) in enumerate(zip(sls, qls)):
        if nq * G > info["dec_rows_max"]:
            for rt in range(-(-nq * G // R)):
                j = (min(R * (rt + 1), nq * G) - 1) // G
                ntk[s, rt] = (sl - nq + j + 1 + 63) // 64
    pieces = {}
    for x in items:
        s, rt, kt0, kt1, slot, q0, nq, sl, qa = (int(v) for v in x[:9])
        assert (q0, nq, sl, qa) == (qsl[s], qls[s], sls[s], sls[s] - qls[s])
        pieces.setdefault((s, rt), []).append((kt0, kt1, slot))
    assert set(pieces) == set(ntk)
    slots = []
    for key, got in pieces.items():
        got.sort()
        if len(got) == 1:
            assert key not in split and got[0][0] == 0 and got[0][1] >= ntk[key] and got[0][2] == -1
            continue
        s0, k = split[key]
        assert k == len(got) and [g[2] for g in got] == list(range(s0, s0 + k))
        assert got[0][0] == 0 and got[-1][1] == ntk[key] and all(a[1] == c[0] and a[0] < a[1] for a, c in zip(got, got[1:]))
        slots += [g[2] for g in got]
    assert len(set(slots)) == len(slots) and all(0 <= v < info["pf_slots_max"] for v in slots)
    if total > info["cus"] // Hkv:
        size = [-(-ntk[int(x[0]), int(x[1])] // len(pieces[int(x[0]), int(x[1])])) for x in items]
        assert all(p >= c for p, c in zip(size, size[1:]))
    assert_close(to_np_f32(out), batch_oracle(b))
