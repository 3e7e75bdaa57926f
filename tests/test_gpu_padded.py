"""GPU: ``gfx906_fa.forward_paged_direct`` reads q and writes its output in
their own [B, Hq, Sq, 128] layout (no copies): every decode row class, both
prefill tile sizes, masks with row tiles split over the keys, transposed
queries, against ``oracle.flat_attention_ref`` on the cache's own values."""
import numpy as np
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, assert_close, need_gpu
from oracle import q8_oracle as O

DEV = "cuda"
pytestmark = pytest.mark.gpu

CASES = [
    # name, seq_lens, Sq, Hq, Hkv, how, q dtype
    ("rows6", [300, 17, 1000], 1, 48, 8, "full", "f32"),
    ("rows30", [700, 40], 5, 6, 1, "causal", "f16"),
    ("rows36_short", [90, 2000], 6, 6, 1, "causal", "bf16"),
    ("rows60_chunks", [500, 130], 10, 6, 1, "causal", "f32"),
    ("rows72", [3000, 64, 900], 12, 48, 8, "causal", "f32"),
    ("rows258_full", [1500, 2600], 43, 48, 8, "full", "f16"),
    ("mask_one_row", [4100], 1, 32, 8, "mask", "f32"),
    ("mask_split", [2500, 900], 9, 8, 1, "mask", "f16"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_padded(case):
    need_gpu()
    name, lens, Sq, Hq, Hkv, how, dt = case
    announce(f"padded {name}")
    B = len(lens)
    b = W.build_batch(lens, [Sq] * B, Hq, Hkv, dtype=dt, seed=sum(map(ord, name)))
    q = b.query.view(B, Sq, Hq, 128).transpose(1, 2)  # a transposed view: copied
    rng = np.random.default_rng(1)
    cols = max(lens) + (1 if name == "mask_split" else 0)
    m = None
    if how == "mask":
        m = rng.standard_normal((B, Sq, cols)).astype(np.float16)
        m[:, :, 70:200] = -np.inf
    off = torch.tensor([n - Sq for n in lens], dtype=torch.int32, device=DEV) if how == "causal" else None
    kp, vp = b.planes()
    args = (kp, vp, b.block_table, b.seq_lens_t, b.scale)
    kw = dict(mask=None if m is None else torch.from_numpy(m).to(DEV), q_abs_offset=off)
    out = gfx906_fa.forward_paged_direct(q, *args, **kw)
    same = gfx906_fa.forward_paged_direct(q.contiguous(), *args, **kw)
    torch.cuda.synchronize()
    assert out.is_contiguous() and out.shape == (B, Hq, Sq, 128) and torch.equal(out, same)
    L = max(lens)
    k = torch.zeros((B, Hkv, L, 128), dtype=b.key.dtype, device=DEV)
    v = torch.zeros_like(k)
    at = 0
    for s, n in enumerate(lens):
        k[s, :, :n] = b.key[at:at + n].transpose(0, 1)
        v[s, :, :n] = b.value[at:at + n].transpose(0, 1)
        at += n
    f = lambda x: x.float().cpu().numpy()  # noqa: E731
    # quantized from the 16-bit values in fp32, as the cache write does
    kq = gfx906_fa.quantize_q8_0(k.contiguous()).cpu().numpy()
    vq = gfx906_fa.quantize_q8_0(v.contiguous()).cpu().numpy()
    ref = O.flat_attention_ref(f(q), kq, O.dequantize_q8_0_rows(vq, 128), b.scale, kv_max=np.asarray(lens),
                               q_abs_offset=None if off is None else off.cpu().numpy(), mask=m)
    assert_close(f(out), ref)
