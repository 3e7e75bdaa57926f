"""GPU: the prefill kernel's 16-byte output stores and its row-wise Q loads on
rows that start on any 2-byte boundary (head stride 131 elements), on both
tile sizes, against the same call on contiguous tensors: bit-identical."""
import math

import numpy as np
import pytest
import torch

import gfx906_fa
import gfx906_fa_workloads as W
from gpu_common import announce, need_gpu

DEV = "cuda"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("q_lens", [[17, 65], [12, 11], [43]], ids=["ks1", "ks2", "rows257"])
def test_prefill_unaligned_rows(q_lens, dtype):
    need_gpu()
    announce(f"prefill unaligned rows {q_lens} {dtype}")
    b = W.build_batch([n + 100 for n in q_lens], q_lens, 48, 8, dtype=dtype, seed=len(q_lens), device=DEV)
    ref = W.attention(b)
    T = b.num_tokens
    q = torch.empty((T, 48, 131), dtype=b.query.dtype, device=DEV)[..., 1:129]
    q.copy_(b.query)
    big = torch.full((T, 48, 131), 7.0, dtype=ref.dtype, device=DEV)
    out = big[..., 1:129]
    b.query = q
    assert W.attention(b, out=out) is out
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    assert bool((big[..., 0] == 7).all()) and bool((big[..., 129:] == 7).all())  # nothing past the rows


def test_noalloc_drops_the_work_list_before_refusing():
    """A batch whose work list no longer fits the allocation-free entry's
    scratch (48 bytes an item), though 20 bytes an item would: it still runs,
    on the 2-D grid, with the outputs of the workspace entry."""
    need_gpu()
    B, Hq, L = 8192, 16, 808
    last = 3                                        # 48 rows: the decode classes are laid out too
    T = (B - 1) * L + last
    info = gfx906_fa.plan_info(B, T, Hq, 1, L, L)
    base, items = info["pf_header_offset"] + 256, info["pf_grid_items"]
    # (the split partials are dropped first; 1 MiB of slack covers the small regions)
    assert base + 48 * items > 64 << 20 and base + 20 * items + (1 << 20) < 64 << 20
    announce(f"noalloc without a work list T={T}")
    g = torch.Generator(device=DEV)
    g.manual_seed(5)
    bs, nb = 16, (L + 15) // 16
    kv = torch.randn((2, L, 1, 128), generator=g, device=DEV, dtype=torch.float16)
    cache = gfx906_fa.new_kv_cache(nb, bs, 1, device=DEV)
    gfx906_fa.reshape_and_cache_q8_kv(kv[0], kv[1], torch.arange(L, device=DEV), cache[:, 0], cache[:, 1])
    bt = torch.arange(nb, dtype=torch.int32, device=DEV).repeat(B, 1)  # every sequence reads the same pages
    lens = np.full(B, L, np.int32)
    lens[-1] = last
    sl = torch.from_numpy(lens).to(DEV)
    qsl = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(DEV)
    q = torch.randn((T, Hq, 128), generator=g, device=DEV, dtype=torch.float16)
    out = torch.empty_like(q)
    Lb = gfx906_fa.lib()
    k, v = cache[:, 0], cache[:, 1]
    p = gfx906_fa._ptr
    scale = 1.0 / math.sqrt(128)
    err = Lb.gfx906_fa_amd_paged_attention_noalloc(
        p(q), 1, q.stride(0), q.stride(1), p(k), p(v), k.stride(0), k.stride(1), p(bt), bt.stride(0), p(sl), p(qsl),
        None, 1, B, T, Hq, 1, 128, bs, L, L, scale, p(out), 1, out.stride(0), out.stride(1),
        gfx906_fa._stream(torch.device(DEV)))
    assert err == 0
    ref = gfx906_fa.paged_attention(q, k, v, bt, sl, qsl, L, L, scale)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
