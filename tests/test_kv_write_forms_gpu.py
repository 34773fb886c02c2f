"""The cache writer's kernels (csrc/atf_kv_write.hip: a few tokens one by one,
pages with one, two or four heads per workgroup) against the CPU model of the
layout and against each other, bit for bit."""
import pytest
import torch

import atflash.ops as ops
import helpers as H
from test_kv_write_gpu import _assemble, _expected_pages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hkv", [(1, 1), (1, 4), (2, 5), (4, 8), (5, 3), (16, 1), (17, 4)])
@pytest.mark.parametrize("start", [-1, 0, 14, 31])
@pytest.mark.parametrize("layout", [0, 1])
def test_few_tokens(n, hkv, start, layout, dev):
    """One to four tokens (the append kernel) and a few more (the page kernel)
    into a cache full of other data: tokens before position 0, past the page
    table's last page and on an invalid entry are skipped, every other slot keeps
    its bits."""
    print(f"[kv_write few] n={n} hkv={hkv} start={start} layout={layout}", flush=True)
    g = torch.Generator().manual_seed(n * 100 + hkv + start)
    k, v = H.randn_bf16((n, hkv, H.D), g), H.randn_bf16((n, hkv, H.D), g)
    pool = 4
    init = (H.randn_bf16((pool, hkv, 16, 16, 8), g), H.randn_bf16((pool, hkv, 128, 16), g))
    for table in ([2, 0, 3], [2, 0], [2, -1, 3], [2, 7, 3]):
        kv = _assemble(*init).to(dev)
        ops.kv_write(kv, k[None].to(dev), v[None].to(dev), torch.tensor([start], dtype=torch.int32, device=dev),
                     torch.tensor([table], dtype=torch.int32, device=dev), None, layout)
        # the tokens that can be placed: the model writes runs of them
        ek, ev = init
        for t in range(n):
            pos = start + t
            if pos >= 0 and pos // 16 < len(table) and 0 <= table[pos // 16] < pool:
                ek, ev = _expected_pages(k[t:t + 1], v[t:t + 1], table, pos, pool, hkv, layout, init=(ek, ev))
        assert torch.equal(kv.cpu(), _assemble(ek, ev)), table


# (rows of tokens x heads at and past each line; heads that divide evenly come first in the grid, others last)
@pytest.mark.parametrize("B,n,hkv", [(1, 300, 1), (2, 3000, 7), (1, 5000, 9), (3, 9000, 5), (1, 70001, 2), (1, 15000, 9),
                                     (2, 5000, 4), (3, 4111, 6), (1, 65536, 8), (2, 43700, 6), (1, 33000, 16)])
def test_forms_agree(B, n, hkv, dev):
    """A call by the two- or four-head kernel (odd head counts: a last group
    partly empty) equals calls of 100 tokens (one head per workgroup) and of 3
    (one by one), RoPE at write, ragged starts."""
    from atflash import rope as R
    print(f"[kv_write forms] B={B} n={n} hkv={hkv}", flush=True)
    _, k, v = H.gpu_qkv(B, n, 1, hkv, dev, seed=n, nq=1)
    starts = torch.tensor([5 + 9 * b for b in range(B)], dtype=torch.int32, device=dev)
    pages = -(-(n + 40) // 16)
    table = torch.randperm(B * pages, generator=torch.Generator().manual_seed(n)).to(torch.int32).view(B, pages).to(dev)
    rt = R.rope_table(n + 40, R.inv_freq(H.D, 1e7, dev))
    whole = torch.zeros((B * pages, hkv, 2, 2048), dtype=torch.bfloat16, device=dev)
    parts = torch.zeros_like(whole)
    ops.kv_write(whole, k, v, starts, table, rt, 0)
    t = 0
    for step in [3] * 20 + [100] * n:
        if t >= n:
            break
        ops.kv_write(parts, k[:, t:t + step], v[:, t:t + step], starts + t, table, rt, 0)
        t += step
    assert torch.equal(whole, parts)


@pytest.mark.parametrize("n,hkv", [(2, 65536), (1, 131080), (1, 131081)])
def test_many_heads(n, hkv, dev):
    """More heads, and more pairs of heads, than a grid's y and z dimensions hold; tokens at the end of one
    page and the start of the next."""
    print(f"[kv_write heads] n={n} hkv={hkv}", flush=True)
    g = torch.Generator(device=dev).manual_seed(hkv)
    k, v = (torch.randn((1, n, hkv, H.D), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    kv = torch.zeros((2, hkv, 2, 2048), dtype=torch.bfloat16, device=dev)
    ops.kv_write(kv, k, v, torch.tensor([15], dtype=torch.int32, device=dev),
                 torch.tensor([[1, 0]], dtype=torch.int32, device=dev), None, 1)
    want = torch.zeros_like(kv)
    for t, (page, slot, v_slot) in enumerate([(1, 15, 15), (0, 0, 0)][:n]):
        want[page, :, 0].view(hkv, 128, 16)[:, :, v_slot] = v[0, t]
        want[page, :, 1].view(hkv, 16, 16, 8)[:, :, slot] = k[0, t].view(hkv, 16, 8)
    assert torch.equal(kv, want)
