"""The batch decode split evenly over the chip (decode_batch_kernel and
decode_merge_kernel<true>, csrc/atf_decode.hip) against the splits by the longest
sequence, which the same call takes with the smaller workspace, and one sequence
of each batch against the oracle.  The lengths choose between three layouts
(short, nearly equal, ragged); max_seq_len only bounds them, so long contexts
need no long sequences here."""
import random

import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


def _lens(kind, B, r):
    if kind == "short":
        return [r.choice((0, 1, 15, 16, 17, 100, 511, 512)) for _ in range(B)]
    if kind == "equal":
        n = r.choice((3000, 4096, 5001))
        return [n - r.randrange(16) for _ in range(B)]
    if kind == "one_long":
        return [r.choice((0, 5, 300)) for _ in range(B - 1)] + [r.choice((20000, 33333))]
    return [int(2 ** r.uniform(0, 13.3)) - 1 for _ in range(B)]  # 0 .. 10000


# batch sizes below, at and past a wave's 64 lanes; runs per kv head 128 to 16
@pytest.mark.parametrize("B,hq,hkv", [(2, 28, 4), (3, 24, 8), (12, 24, 8), (31, 16, 16), (64, 14, 2), (65, 8, 4),
                                      (100, 32, 4), (255, 16, 1)])
@pytest.mark.parametrize("kind", ["short", "equal", "one_long", "ragged"])
def test_even_split(kind, B, hq, hkv, dev):
    from atflash import _lib, atflash_window as AW, fiwin_common as FW, interface, rope as R
    from atflash.cache import PagedKVCache
    L = _lib.lib()
    base = 1e7
    r = random.Random(f"{kind}{B}{hkv}")
    lens = _lens(kind, B, r)
    if sum(lens) > 400_000:
        lens = [n // 4 for n in lens]
    maxlen = max(max(lens), 98304 * 16 // (B * hkv) + 16)
    small, even = (f(B, hq, hkv, maxlen) for f in (L.atf_decode_workspace_bytes, L.atf_decode_workspace_bytes_even))
    assert even == hkv * (256 // hkv) * 2 * 16 * 130 * 4 > small or (B * hkv >= 512 and even == small)
    width = -(-maxlen // 16)
    need = [-(-n // 16) for n in lens]
    cache = PagedKVCache(sum(need) + 1, hkv, dev)
    cache._free = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(B)).tolist()
    for b, n in enumerate(lens):
        cache.add_sequence(b, n)
    table = cache.page_table(list(range(B)), width)
    rt = R.rope_table(maxlen, R.inv_freq(H.D, base, dev))
    total = max(sum(lens), 1)
    _, k, v = H.gpu_qkv(1, total, 1, hkv, dev, seed=B, nq=1)
    at, probe = 0, None
    for b, n in enumerate(lens):
        if n:
            torch.ops.atflash.kv_write(cache.kv, k[:, at:at + n], v[:, at:at + n],
                                       torch.zeros(1, dtype=torch.int32, device=dev), table[b:b + 1].contiguous(), rt, 0)
            if probe is None or (n > 300 and lens[probe[0]] <= 300):
                probe = (b, at)
            at += n
    q = H.gpu_qkv(B, 1, hq, 1, dev, seed=B + 1, nq=1)[0][:, 0].contiguous()
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    for name, z in (("off", None), ("level", AW.window_zhi_from_kret(H.D, base, 2.0, 1 << 20)),
                    ("vec8", FW.zhi_slice_vec8(H.D, base, 2.0).tolist())):
        print(f"[even split] {kind} B={B} hkv={hkv} max {max(lens)} {name}", flush=True)
        out = interface.decode_paged(q, cache, table, seq, maxlen, zhi=z, rope=rt)
        ref = torch.empty_like(out)
        ws = torch.empty(small // 4 + 4, dtype=torch.float32, device=dev)
        n = 16 if name == "vec8" else 8
        entry = L.atf_decode_paged_slices_bf16 if n == 16 else L.atf_decode_paged_bf16
        _lib.check(entry(ref.data_ptr(), hq * H.D, H.D, q.data_ptr(), hq * H.D, H.D, cache.kv.data_ptr(),
                         cache.num_pages, table.data_ptr(), width, seq.data_ptr(), B, hq, hkv, maxlen,
                         _lib.zhi_array(z, n), H.D ** -0.5, rt.data_ptr(), rt.shape[0], 0, ws.data_ptr(), small,
                         _lib.stream_of(dev)))
        empty = [b for b in range(B) if lens[b] == 0]
        assert torch.equal(out[empty], torch.zeros_like(out[empty]))
        # the same fp32 partial sums in other groups, rounded to bf16 once: one unit in the last place of each
        # value, and of the probabilities' bf16 rounding against another reference max (2^-9 of sum |p v|)
        assert torch.isfinite(out).all()
        assert torch.allclose(out.float(), ref.float(), rtol=2 ** -7, atol=4e-3), (out.float() - ref.float()).abs().max()
        if probe is not None and lens[probe[0]] <= 12000:
            b, a0 = probe
            kc, vc = k[0, a0:a0 + lens[b]].cpu(), v[0, a0:a0 + lens[b]].cpu()
            if name == "vec8":
                o = H.decode_oracle_vec8(q[b].cpu(), kc, vc, base, z, True)
            else:
                o = H.decode_oracle(q[b].cpu(), kc, vc, base, 2.0 if z else float("inf"), True)
            H.assert_close(out[b], o, f"sequence {b} ({lens[b]} tokens) {name}")
