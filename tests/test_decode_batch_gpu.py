"""The batch decode spread over the chip wave by wave (decode_wave_kernel and its
merge kernels, csrc/atf_decode.hip).  It has to give the bits of the splits by the
longest sequence (decode_kernel, decode_merge_kernel), which the same call takes with
the smaller workspace: a page left out or read twice, a partial of another
sequence or an old one would show in them.  So a sequence's bits do not depend on the
other sequences' lengths either.  One sequence of each batch is checked against the
oracle.  max_seq_len only bounds the lengths, so long contexts need no long sequences
here."""
import random

import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

PAGES = 200_000  # of the batch if every sequence were as long as the longest: past the rule's lines


def _lens(kind, B, r):
    if kind == "short":
        return [r.choice((0, 1, 15, 16, 17, 100, 511, 512)) for _ in range(B)]
    if kind == "equal":
        n = r.choice((3000, 4096, 5001))
        return [n - r.randrange(16) for _ in range(B)]
    if kind == "one_long":
        return [r.choice((0, 5, 300)) for _ in range(B - 1)] + [r.choice((20000, 33333))]
    return [int(2 ** r.uniform(0, 13.3)) - 1 for _ in range(B)]  # 0 .. 10000


# 16 to 511 (sequence, kv head) pairs, so 16 to 1 splits; batch sizes below, at and past the 64 lanes that
# rank a batch's lengths; waves that fit the chip at once (4 x 4 and 64 x 2 pairs) and more
@pytest.mark.parametrize("B,hq,hkv", [(4, 28, 4), (3, 24, 8), (12, 32, 2), (12, 24, 8), (31, 16, 16), (64, 14, 2),
                                      (65, 8, 4), (100, 32, 4), (255, 16, 1), (511, 4, 1)])
@pytest.mark.parametrize("kind", ["short", "equal", "one_long", "ragged"])
def test_spread_batch(kind, B, hq, hkv, dev):
    from atflash import _lib, atflash_window as AW, fiwin_common as FW, interface, rope as R
    from atflash.cache import PagedKVCache
    L = _lib.lib()
    base = 1e7
    r = random.Random(f"{kind}{B}{hkv}")
    lens = _lens(kind, B, r)
    if sum(lens) > 400_000:
        lens = [n // 4 for n in lens]
    width = max(-(-PAGES // (B * hkv)), -(-max(lens) // 16))
    maxlen = width * 16
    small, even = (f(B, hq, hkv, maxlen) for f in (L.atf_decode_workspace_bytes, L.atf_decode_workspace_bytes_even))
    assert even == B * hkv * -(-256 // (B * hkv)) * 8 * (hq // hkv) * 130 * 4 > small
    need = [-(-n // 16) for n in lens]
    cache = PagedKVCache(sum(need) + 1, hkv, dev)
    cache._free = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(B)).tolist()
    for b, n in enumerate(lens):
        cache.add_sequence(b, n)
    table = cache.page_table(list(range(B)), width)
    rt = R.rope_table(maxlen, R.inv_freq(H.D, base, dev))
    _, k, v = H.gpu_qkv(1, max(sum(lens), 1), 1, hkv, dev, seed=B, nq=1)
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

    def decode(z, n, nbytes, lengths):
        out = torch.empty_like(q)
        ws = torch.full((nbytes // 4 + 4,), float("nan"), dtype=torch.float32, device=dev)
        entry = L.atf_decode_paged_slices_bf16 if n == 16 else L.atf_decode_paged_bf16
        _lib.check(entry(out.data_ptr(), hq * H.D, H.D, q.data_ptr(), hq * H.D, H.D, cache.kv.data_ptr(),
                         cache.num_pages, table.data_ptr(), width, lengths.data_ptr(), B, hq, hkv, maxlen,
                         _lib.zhi_array(z, n), H.D ** -0.5, rt.data_ptr(), rt.shape[0], 0, ws.data_ptr(), nbytes,
                         _lib.stream_of(dev)))
        return out

    for name, z in (("off", None), ("level", AW.window_zhi_from_kret(H.D, base, 2.0, 1 << 20)),
                    ("vec8", FW.zhi_slice_vec8(H.D, base, 2.0).tolist())):
        print(f"[spread batch] {kind} B={B} hkv={hkv} max {max(lens)} {name}", flush=True)
        n = 16 if name == "vec8" else 8
        out = decode(z, n, even, seq)
        assert torch.equal(out, decode(z, n, small, seq))
        assert torch.equal(out, interface.decode_paged(q, cache, table, seq, maxlen, zhi=z, rope=rt))
        assert torch.isfinite(out).all()
        empty = [b for b in range(B) if lens[b] == 0]
        assert torch.equal(out[empty], torch.zeros_like(out[empty]))
        if probe is not None:
            b, a0 = probe
            alone = torch.zeros_like(seq)
            alone[b] = seq[b]
            assert torch.equal(out[b], decode(z, n, even, alone)[b])
            # (of a few tokens the outputs are near 1, where rounding them to bf16 alone is off by 2^-10, the bar, on average)
            if 100 <= lens[b] <= 12000:
                kc, vc = k[0, a0:a0 + lens[b]].cpu(), v[0, a0:a0 + lens[b]].cpu()
                if name == "vec8":
                    o = H.decode_oracle_vec8(q[b].cpu(), kc, vc, base, z, True)
                else:
                    o = H.decode_oracle(q[b].cpu(), kc, vc, base, 2.0 if z else float("inf"), True)
                H.assert_close(out[b], o, f"sequence {b} ({lens[b]} tokens) {name}")
