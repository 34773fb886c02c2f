"""The decode over contiguous K and V rows (decode_rows_kernel, csrc/atf_decode.hip)
against the fp32 oracle and, bit for bit, against the packed paged cache: every table kind,
both layouts, RoPE on and off, NHD and HND strides, token counts at the edges of
a 16-token block, of a wave's group and of a split, GQA groups up to 16."""
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

TABLES = ["off", "level", "vec8"]


def _table(name, base, k_ret):
    from atflash import atflash_window as AW, fiwin_common as FW
    if name == "off":
        return None
    if name == "level":
        return list(AW.window_zhi_from_kret(H.D, base, k_ret, 1 << 20))
    return FW.zhi_slice_vec8(H.D, base, k_ret).tolist()


@pytest.mark.parametrize("N,hq,hkv", [(1, 7, 1), (15, 4, 4), (16, 6, 2), (17, 28, 4), (33, 16, 1), (511, 12, 4),
                                      (513, 24, 8), (4097, 28, 4), (9000, 18, 2)])
@pytest.mark.parametrize("layout,rope", [("half_split", True), ("half_split", False), ("sorted_pair", False)])
def test_rows_decode(N, hq, hkv, layout, rope, dev):
    from atflash import interface as I, ops, rope as R
    base, k_ret = 1e4, 0.5  # widths 3 .. 270: boundaries inside the pages and inside the lengths
    g = torch.Generator().manual_seed(N * 31 + hq)
    q, k, v = (H.randn_bf16(s, g) for s in ((hq, H.D), (N, hkv, H.D), (N, hkv, H.D)))
    rt = R.rope_table(N, R.inv_freq(H.D, base, dev)) if rope else None
    for name in TABLES:
        print(f"[rows decode] N={N} hq={hq} hkv={hkv} {layout} rope={rope} {name}", flush=True)
        z = _table(name, base, k_ret)
        out = I.single_decode_with_kv_cache(q.to(dev), k.to(dev), v.to(dev), maybe_zhi=z, rope=rt, layout=layout)
        # HND strides, and rows inside wider ones (a fused qkv projection's output)
        hnd = I.single_decode_with_kv_cache(q.to(dev), k.transpose(0, 1).contiguous().to(dev),
                                            v.transpose(0, 1).contiguous().to(dev), maybe_zhi=z, kv_layout="HND",
                                            rope=rt, layout=layout)
        wide = torch.cat([k, v], dim=-1).to(dev)
        w = I.single_decode_with_kv_cache(q.to(dev), wide[..., :H.D], wide[..., H.D:], maybe_zhi=z, rope=rt,
                                          layout=layout)
        assert torch.equal(out, hnd) and torch.equal(out, w), "strides"
        # the packed path: the same operands in the same order
        kvc, table = I.pack_kv(k[None].to(dev), v[None].to(dev), rope=rt, layout=layout)
        seq = torch.tensor([N], dtype=torch.int32, device=dev)
        packed = ops.decode_paged(q[None].to(dev), kvc, table, seq, N, z, H.D ** -0.5, rt, I._layout_id(layout))[0]
        assert torch.equal(out, packed), "packed"
        if layout == "half_split":
            if name == "vec8":
                ref = H.decode_oracle_vec8(q, k, v, base, z, rope)
            else:
                ref = H.decode_oracle(q, k, v, base, k_ret if z else float("inf"), rope)
            H.assert_close(out, ref, f"N={N} {name}")


def test_rows_decode_batch_and_refusals(dev):
    """A batch equals its sequences alone, bit for bit where the split is the
    same; token strides past the kernel's addressing go through the pages; what
    the kernel cannot take raises."""
    from atflash import interface as I, ops
    _, k, v = H.gpu_qkv(3, 300, 1, 4, dev, seed=5, nq=1)
    q = H.gpu_qkv(3, 1, 8, 1, dev, seed=6, nq=1)[0][:, 0]
    out = I.decode_contiguous(q, k, v, None, H.D ** -0.5, None, 0)
    for b in range(3):
        assert torch.equal(out[b], I.single_decode_with_kv_cache(q[b], k[b], v[b]))
    one = torch.as_strided(k, (1, 1, 4, H.D), (k.stride(0), (1 << 26) + 8, H.D, 1))
    assert ops.decode_rows(q[:1], one, one, None, H.D ** -0.5, None, 0) is None
    assert torch.allclose(I.decode_contiguous(q[:1], one, one, None, H.D ** -0.5, None, 0).float(),
                          k[:1, :1].float().repeat_interleave(2, dim=2)[:, 0], rtol=2 ** -7, atol=0)
    for bad_k in (k.float(), k[..., :64], k[:, :, :3]):
        with pytest.raises((ValueError, RuntimeError)):
            I.decode_contiguous(q, bad_k, bad_k, None, H.D ** -0.5, None, 0)
    with pytest.raises(ValueError):  # 8-byte aligned rows
        flat = torch.empty(k.numel() + 8, dtype=torch.bfloat16, device=dev)
        I.decode_contiguous(q, flat[4:4 + k.numel()].view(k.shape), v, None, H.D ** -0.5, None, 0)
    with pytest.raises(ValueError):
        I.decode_contiguous(q, k[:, :0], v[:, :0], None, H.D ** -0.5, None, 0)
