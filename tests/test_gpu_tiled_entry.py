"""GPU: the C entry ``gfx906_fa_amd_paged_attention_tiled`` (no workspace, every
sequence through the 256-row tiled kernel on a 2-D grid) over planar Q8 V and,
after ``gfx906_fa_amd_pack_flat_kv``, over planar fp16 V: ragged query counts
(none included), pages of one, three and four sub-pages and one page per
sequence, page windows that slide (more than 64 and 128 key tiles), causal
bounds given and derived, masks of fewer and more columns than keys at both
load widths, every query type, against ``oracle.flat_attention_ref``."""
import numpy as np
import pytest
import torch

import gfx906_fa
from gpu_common import announce, assert_close, need_gpu
from oracle import q8_oracle as O

DEV = "cuda"
pytestmark = pytest.mark.gpu
DT = {"f32": (0, torch.float32), "f16": (1, torch.float16), "bf16": (2, torch.bfloat16)}

CASES = [
    # name, V format, heads, page tokens (0: one page), keys, query tokens, how, mask columns, query type
    ("q8_full_page16", 0, (8, 4), 16, [1, 15, 64, 65], [1, 3, 129, 2], "full", 0, "f32"),
    ("q8_causal_page48", 0, (6, 1), 48, [4200, 47, 49, 300], [43, 47, 0, 86], "causal", 0, "f16"),
    ("q8_offset_page64", 0, (3, 3), 64, [130, 500], [40, 300], "offset", 0, "bf16"),
    ("q8_causal_two_slides", 0, (2, 1), 48, [8300], [12], "causal", 0, "f32"),
    ("q8_mask_fewer_cols", 0, (6, 1), 48, [200, 4111], [5, 43], "mask", 160, "f16"),
    ("q8_mask_odd_cols", 0, (8, 1), 16, [70, 33], [33, 17], "mask", 75, "bf16"),
    ("f16_full", 1, (8, 4), 0, [1, 16, 100, 256], [2, 65, 129, 1], "full", 0, "f32"),
    ("f16_causal_slide", 1, (6, 1), 0, [4200, 129, 4150], [43, 129, 7], "causal", 0, "bf16"),
    ("f16_offset_two_slides", 1, (2, 2), 0, [8300, 8193], [3, 140], "offset", 0, "f16"),
    ("f16_mask", 1, (4, 2), 0, [500, 4120], [130, 9], "mask", 4124, "f32"),
    ("f16_mask_odd_cols", 1, (6, 2), 0, [90, 64], [20, 43], "mask", 91, "f16"),
    ("f16_mask_bf16_query", 1, (6, 1), 0, [65], [50], "mask", 64, "bf16"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tiled_entry(case):
    need_gpu()
    name, vf, (Hq, Hkv), bs, lens, nqs, how, cols, dt = case
    announce(f"tiled entry {name}")
    code, td = DT[dt]
    rng = np.random.default_rng(sum(map(ord, name)))
    B, T, L = len(lens), sum(nqs), max(lens)
    scale = 0.09
    q = torch.from_numpy(rng.standard_normal((T, Hq, 128)).astype(np.float32)).to(td).to(DEV)
    k = rng.standard_normal((B, Hkv, L, 128)).astype(np.float16)
    v = rng.standard_normal((B, Hkv, L, 128)).astype(np.float16)
    kq = O.quantize_q8_0_rows(k)
    lib, p, st = gfx906_fa.lib(), gfx906_fa._ptr, gfx906_fa._stream(torch.device(DEV, torch.cuda.current_device()))
    dev = lambda x: None if x is None else torch.from_numpy(x).to(DEV)  # noqa: E731
    if vf == 1:  # one page per sequence
        vref, skp = v, (L + 15) // 16
        kp = torch.empty((B, Hkv, skp * 2176), dtype=torch.uint8, device=DEV)
        vp = torch.empty((B, Hkv, skp * 4096), dtype=torch.uint8, device=DEV)
        kd, vd = dev(kq), dev(v)
        assert lib.gfx906_fa_amd_pack_flat_kv(p(kd), p(vd), p(kp), p(vp), B * Hkv, L, 128, st) == 0
        bs, bt = skp * 16, np.arange(B, dtype=np.int32)[:, None]
    else:
        vref = O.dequantize_q8_0_rows(O.quantize_q8_0_rows(v), 128)
        nb = (L + bs - 1) // bs
        bt = rng.permutation(B * nb).astype(np.int32).reshape(B, nb)
        cache = gfx906_fa.new_kv_cache(B * nb, bs, Hkv, device=DEV)
        kp, vp = cache[:, 0], cache[:, 1]
        pos = np.arange(L)
        for b in range(B):
            slots = dev(bt[b, pos // bs].astype(np.int64) * bs + pos % bs)
            gfx906_fa.reshape_and_cache_q8_kv(dev(k[b].transpose(1, 0, 2).copy()), dev(v[b].transpose(1, 0, 2).copy()),
                                              slots, kp, vp)
    qa = np.array([n - m - 20 for n, m in zip(lens, nqs)], np.int32) if how == "offset" else None
    mask = None
    if how == "mask":
        mask = rng.standard_normal((B, max(nqs), cols)).astype(np.float16)
        mask[:, ::3, :cols // 2] = -np.inf
    out = torch.full((T, Hq, 128), 7.0, dtype=torch.float32, device=DEV)
    btd, sl, md, qad = dev(bt), dev(np.asarray(lens, np.int32)), dev(mask), dev(qa)
    qsl = dev(np.concatenate([[0], np.cumsum(nqs)]).astype(np.int32))
    err = lib.gfx906_fa_amd_paged_attention_tiled(
        p(q), code, q.stride(0), q.stride(1), p(kp), p(vp), vf, kp.stride(0), kp.stride(1), vp.stride(0), vp.stride(1),
        p(btd), btd.stride(0), p(sl), p(qsl), p(qad), 1 if how in ("causal", "offset") else 0, p(md),
        0 if mask is None else md.stride(0), 0 if mask is None else md.stride(1), cols, B, T, Hq, Hkv, 128, bs,
        max(nqs), scale, p(out), out.stride(0), out.stride(1), st)
    assert err == 0
    torch.cuda.synchronize()
    qf, got, at = q.float().cpu().numpy(), out.cpu().numpy(), 0
    for b, (n, m) in enumerate(zip(lens, nqs)):
        if m:
            off = None if how in ("full", "mask") else np.array([n - m if qa is None else qa[b]], np.int32)
            mb = None
            if mask is not None:  # columns past the mask add 0
                mb = np.zeros((1, m, max(n, cols)), np.float16)
                mb[0, :, :cols] = mask[b, :m]
            ref = O.flat_attention_ref(qf[at:at + m].transpose(1, 0, 2)[None], kq[b:b + 1, :, :n], vref[b:b + 1, :, :n],
                                       scale, q_abs_offset=off, mask=mb)
            assert_close(got[at:at + m].transpose(1, 0, 2)[None], ref)
        at += m


def test_tiled_entry_refuses():
    """Unsupported configurations are errors before anything is launched."""
    need_gpu()
    lib = gfx906_fa.lib()
    x = torch.zeros(1 << 16, dtype=torch.uint8, device=DEV)
    base = x.data_ptr()

    def call(vf=0, hq=2, hkv=1, d=128, bs=16, code=0, koff=0, cols=0, mask=None):
        return lib.gfx906_fa_amd_paged_attention_tiled(
            base, code, 256, 128, base + koff, base, vf, 2176, 2176, 2176, 2176, base, 1, base, base, None, 0, mask, 0, 0,
            cols, 1, 1, hq, hkv, d, bs, 1, 0.1, base, 256, 128, None)

    for bad in (dict(vf=2), dict(hq=3, hkv=2), dict(d=64), dict(bs=24), dict(code=3), dict(koff=8),
                dict(mask=base, cols=-1)):
        assert call(**bad) != 0, bad
