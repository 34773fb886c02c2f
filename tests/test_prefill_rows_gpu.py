"""Q in and O out in whole rows (csrc/atf_prefill.hip: q_request, store_rows), in
both prefill kernels: an output that is only 8-byte aligned, with gaps between
its rows, gets the bits of a dense one, and nothing between its rows changes."""
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,rope", [(0, True), (0, False), (1, False)])  # RoPE is fused for half-split only
@pytest.mark.parametrize("n", [1, 7, 33, 129, 1283])  # 1283 x 28 heads: the 256-row kernel
def test_output_rows_8_byte_aligned(n, layout, rope, dev):
    from atflash import _lib, interface as I, ops, rope as R
    hq, hkv, pitch = 28, 4, H.D + 4
    q, k, v = H.gpu_qkv(1, n, hq, hkv, dev, seed=29)
    q = torch.nn.functional.pad(q, (8, 0))[..., 8:]  # rows of 136 elements, 16-byte aligned
    rt = R.rope_table(n, R.inv_freq(H.D, 1e4, dev)) if rope else None
    kvc, table = I.pack_kv(k, v, rope=rt, layout=("half_split", "sorted_pair")[layout])
    ref, lse = ops.prefill(q, kvc, table, n, 0, None, H.D ** -0.5, rt, layout)
    buf = torch.full((n * hq * pitch + 4,), 7.0, dtype=torch.bfloat16, device=dev)
    lse2 = torch.empty_like(lse)
    _lib.check(_lib.lib().atf_prefill_bf16(
        buf.data_ptr() + 8, n * hq * pitch, hq * pitch, pitch, lse2.data_ptr(), q.data_ptr(), *q.stride()[:3],
        kvc.data_ptr(), kvc.shape[0], table.data_ptr(), table.shape[1],
        1, n, n, 0, hq, hkv, None, H.D ** -0.5, _lib.ptr(rt), n if rope else 0, layout, _lib.stream_of(q.device)))
    rows = buf[4:].view(1, n, hq, pitch)
    assert torch.equal(rows[..., :H.D], ref) and torch.equal(lse2, lse)
    assert (buf[:4] == 7).all() and (rows[..., H.D:] == 7).all()
    # the last rows against fp32 attention (window off) on the CPU
    r = max(0, n - 40)
    qf, kf, vf = q.cpu(), k.cpu(), v.cpu().float()
    qf, kf = (H.rotate(t, torch.arange(n), 1e4) if rope else t.float() for t in (qf, kf))
    s = torch.einsum("qhd,khd->hqk", qf[0, r:], kf[0].repeat_interleave(hq // hkv, 1)) * H.D ** -0.5
    s = s.masked_fill(torch.arange(n)[None, :] > torch.arange(r, n)[:, None], float("-inf"))
    want = torch.einsum("hqk,khd->qhd", s.softmax(-1), vf[0].repeat_interleave(hq // hkv, 1))
    H.assert_close(rows[:, r:, :, :H.D], want[None], f"rows {r}..{n}")
