"""The prefill's two kernels (csrc/atf_prefill.hip): launches whose 128-row
workgroups fit the chip at once take the one-wave-per-SIMD kernel, larger ones
the 256-row kernel.  Both form every sum in the same order, so a chunk by the
first equals the same rows of a single shot by the second, bit for bit."""
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

N, HQ, HKV = 3000, 28, 4  # 24 tiles of 128 rows x 28 heads: more than 256 workgroups


@pytest.mark.parametrize("rope", [True, False])
@pytest.mark.parametrize("k_ret", [None, 0.02, 2.0])
@pytest.mark.parametrize("growing", [False, True])
def test_chunks_equal_single_shot(rope, k_ret, growing, dev):
    """Chunks of 1 to 1100 rows at offsets 0 to 2976 (diagonals anywhere in a tile
    pair, rows past the queries, a partial last page), level boundaries inside
    tile pairs (k = 0.02), and scores that outgrow the reference max again and
    again (the rescale path of both kernels)."""
    from atflash import atflash_window as AW, interface as I, ops, rope as R
    base = 1e4
    q, k, v = H.gpu_qkv(1, N, HQ, HKV, dev, seed=17)
    if growing:
        k = (k.float() * torch.linspace(0.2, 12.0, N, device=dev)[None, :, None, None]).to(torch.bfloat16)
    zhi = None if k_ret is None else list(AW.window_zhi_from_kret(H.D, base, k_ret, 1 << 20))
    rt = R.rope_table(N, R.inv_freq(H.D, base, dev)) if rope else None
    kvc, table = I.pack_kv(k, v, rope=rt)
    perm = torch.randperm(table.shape[1], generator=torch.Generator().manual_seed(3)).to(dev)
    shuffled = torch.empty_like(kvc)
    shuffled[perm] = kvc  # scattered pages
    table = perm.to(torch.int32)[None].contiguous()
    run = lambda a, n: ops.prefill(q[:, a:a + n], shuffled, table, a + n, a, zhi, H.D ** -0.5, rt, 0)  # noqa: E731
    out, lse = run(0, N)
    if k_ret == 2.0 and not growing:
        rows = {r: q[:, r:r + 32].cpu() for r in (0, 1504, 2944)}
        ref = H.prefill_oracle_rows(rows, k.cpu(), v.cpu(), base, k_ret, sorted(rows), rope=rope)
        for r in rows:
            H.assert_close(out[:, r:r + 32], ref[r], f"rows {r}")
    for a, n in ((0, 1), (0, 32), (0, 33), (0, 127), (0, 129), (32, 100), (96, 64), (128, 128), (160, 257), (1024, 1),
                 (1024, 1100), (1920, 1000), (2976, 24), (2912, 88), (1888, 1112)):
        print(f"[prefill solo] rope={rope} k={k_ret} growing={growing} rows {a}..{a + n}", flush=True)
        o, l = run(a, n)
        assert torch.equal(o, out[:, a:a + n]) and torch.equal(l, lse[:, :, a:a + n]), (a, n)


def test_missing_pages(dev):
    """An entry outside the pool reads as a page of zeros in both kernels."""
    from atflash import interface as I, ops
    q, k, v = H.gpu_qkv(1, N, HQ, HKV, dev, seed=23)
    k[:, 320:336], v[:, 320:336], k[:, 1600:1616], v[:, 1600:1616] = 0, 0, 0, 0
    kvc, table = I.pack_kv(k, v)
    full = ops.prefill(q, kvc, table, N, 0, None, H.D ** -0.5, None, 0)
    table[0, 20], table[0, 100] = -1, kvc.shape[0]
    for a, n in ((0, N), (1984, 512)):
        o, l = ops.prefill(q[:, a:a + n], kvc, table, a + n, a, None, H.D ** -0.5, None, 0)
        assert torch.equal(o, full[0][:, a:a + n]) and torch.equal(l, full[1][:, :, a:a + n])
