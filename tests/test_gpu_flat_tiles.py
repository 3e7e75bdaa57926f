"""GPU: ``gfx906_fa.forward`` past the decode shapes (more than 16 rows per
kv-head, or a mask): K and V dequantized once into tile images, row tiles
split over the keys.  Key counts around the 64-key tile and the split, ragged
kv_max (0 keys included), both mask load widths, inputs whose bases miss the
wide loads' alignment, and more batch rows than the work list takes, against
``oracle.flat_attention_ref``."""
import numpy as np
import pytest
import torch

import gfx906_fa
from gpu_common import announce, assert_close, need_gpu
from oracle import q8_oracle as O

DEV = "cuda"
pytestmark = pytest.mark.gpu

CASES = [
    # name, B, Hq, Hkv, Sq, Skv, kv_max, q_abs, mask columns, offset of the K / V bases in elements
    ("one_key", 1, 8, 4, 17, 1, None, None, None, 0),
    ("skv63", 2, 8, 4, 20, 63, None, None, None, 0),
    ("skv64_odd_base", 1, 6, 1, 64, 64, None, [0], None, 1),
    ("skv65_rows257", 2, 6, 1, 43, 65, [65, 0], None, None, 0),
    ("split_causal", 1, 8, 4, 129, 2047, None, [1918], None, 0),
    ("split_full_kvmax", 2, 4, 2, 70, 3001, [3001, 1111], None, None, 4),
    ("mask_split", 1, 8, 1, 9, 2050, None, None, 2052, 0),
    ("mask_decode_rows", 2, 8, 8, 1, 1500, [1500, 700], None, 1501, 0),
    ("many_rows_no_list", 8200, 2, 2, 17, 20, None, None, None, 0),
]


def _at(x, off):
    """x on the device, its first element `off` elements past an aligned base."""
    buf = torch.empty(x.size + off, dtype=torch.from_numpy(x[:0]).dtype, device=DEV)
    buf[off:].copy_(torch.from_numpy(x).reshape(-1))
    return buf[off:].view(x.shape)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_forward_tiles(case):
    need_gpu()
    name, B, Hq, Hkv, Sq, Skv, kvm, qa, cols, off = case
    announce(f"forward tiles {name}")
    rng = np.random.default_rng(sum(map(ord, name)))
    q = rng.standard_normal((B, Hq, Sq, 128)).astype(np.float32)
    kq = O.quantize_q8_0_rows(rng.standard_normal((B, Hkv, Skv, 128)).astype(np.float16))
    v = rng.standard_normal((B, Hkv, Skv, 128)).astype(np.float16)
    m = None if cols is None else rng.standard_normal((B, Sq, cols)).astype(np.float16)
    if m is not None:
        m[:, ::3, : Skv // 2] = -np.inf    # whole pieces of these rows see nothing
        m[:, 1::3, Skv // 2:Skv] = np.finfo(np.float16).min
    kvm = None if kvm is None else np.asarray(kvm, np.int32)
    qa = None if qa is None else np.asarray(qa, np.int32)
    dev = lambda x: None if x is None else torch.from_numpy(x).to(DEV)  # noqa: E731
    out = gfx906_fa.forward(dev(q), _at(kq, off), _at(v, off), 0.09, kv_max=dev(kvm), mask=dev(m),
                            q_abs_offset=dev(qa))
    torch.cuda.synchronize()
    assert out.is_contiguous() and out.shape == q.shape
    assert_close(out.cpu().numpy(), O.flat_attention_ref(q, kq, v, 0.09, kv_max=kvm, q_abs_offset=qa, mask=m))


UNSEEN = [
    # name, B, Hq, Hkv, Sq, Skv, kv_max, q_abs, masked, first key with bad bytes, query tokens compared
    ("kv_max", 4, 8, 4, 20, 200, [16, 48, 112, 70], None, False, None, 20),
    ("kv_max_one_tile", 2, 6, 1, 3, 64, [16, 63], None, False, None, 3),
    ("kv_max_split", 2, 8, 4, 70, 3001, [1120, 1111], None, False, None, 70),
    ("causal_end", 2, 8, 4, 40, 200, None, [8, 30], False, None, 40),
    ("causal_end_split", 1, 8, 4, 129, 2047, None, [1500], False, None, 129),
    ("mask", 2, 8, 1, 9, 200, [96, 33], None, True, None, 9),
    ("mask_split", 1, 8, 1, 9, 2050, [1969], None, True, None, 9),
    ("earlier_row_tile", 1, 64, 8, 64, 64, None, [0], False, 32, 32),  # 32 query tokens a row tile
    ("no_list", 8200, 2, 2, 17, 20, 16, None, False, None, 17),
    ("decode_rows", 4, 8, 4, 1, 200, [16, 48, 112, 64], None, False, None, 1),
]


@pytest.mark.parametrize("case", UNSEEN, ids=[c[0] for c in UNSEEN])
def test_forward_unseen_keys(case):
    """Inf and NaN in the V rows and K scales of keys past a row tile's last
    visible one (a buffer larger than its context) leave the output as it is
    with zeros there, bit for bit."""
    need_gpu()
    name, B, Hq, Hkv, Sq, Skv, kvm, qa, masked, first, ntok = case
    announce(f"forward unseen keys {name}")
    rng = np.random.default_rng(sum(map(ord, name)))
    q = rng.standard_normal((B, Hq, Sq, 128)).astype(np.float32)
    kq = O.quantize_q8_0_rows(rng.standard_normal((B, Hkv, Skv, 128)).astype(np.float16))
    v = rng.standard_normal((B, Hkv, Skv, 128)).astype(np.float16)
    m = rng.standard_normal((B, Sq, Skv)).astype(np.float16) if masked else None
    kvm = None if kvm is None else np.broadcast_to(np.asarray(kvm, np.int32), (B,)).copy()
    qa = None if qa is None else np.asarray(qa, np.int32)
    bad_k, bad_v = kq.copy(), v.copy()
    for b in range(B):
        end = Skv if kvm is None else int(kvm[b])
        end = end if qa is None else min(end, int(qa[b]) + Sq)
        end = end if first is None else first
        kq[b, :, end:] = 0
        v[b, :, end:] = 0
        bad_v[b, :, end:, 0::2] = np.nan
        bad_v[b, :, end:, 1::2] = np.inf
        bad_k[b, :, end:].reshape(Hkv, Skv - end, 4, 34)[..., :2] = np.array([0xFF, 0x7F], np.uint8)  # a NaN scale
    dev = lambda x: None if x is None else torch.from_numpy(x).to(DEV)  # noqa: E731
    out, ref = (gfx906_fa.forward(dev(q), dev(k_), dev(v_), 0.09, kv_max=dev(kvm), mask=dev(m), q_abs_offset=dev(qa))
                for k_, v_ in ((bad_k, bad_v), (kq, v)))
    torch.cuda.synchronize()
    assert torch.equal(out[:, :, :ntok], ref[:, :, :ntok])
    want = O.flat_attention_ref(q, kq, v, 0.09, kv_max=kvm, q_abs_offset=qa, mask=m)
    assert_close(ref.cpu().numpy()[:, :, :ntok], want[:, :, :ntok])
