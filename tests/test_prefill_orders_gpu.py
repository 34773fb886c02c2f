"""The prefill's block order (csrc/atf_prefill.hip: prefill_block): (query tile,
sequence, kv head) units dealt out over the XCDs.  Every row of every head of
every sequence must be written once, whatever the counts: the outputs are
compared with the oracle, and a batch bit for bit with its sequences run alone."""
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,hq,hkv", [
    (1, 33, 3, 1),     # one unit
    (3, 700, 14, 2),   # 3 tiles: 18 units, a partial last round
    (5, 257, 6, 3),    # the second tile of one row; 30 units
    (1, 2304, 8, 2),   # 9 tiles: a partial second round
    (2, 1024, 16, 1),  # GQA group 16: 8 units, one round
])
def test_block_order(B, N, hq, hkv, dev):
    from atflash import atflash_window as AW, interface, rope as R
    base, k_ret = 1e7, 0.5
    print(f"[prefill order] B={B} N={N} hq={hq} hkv={hkv}", flush=True)
    q, k, v = H.qkv(B, N, hq, hkv, seed=N + hq)
    zhi = AW.window_zhi_from_kret(H.D, base, k_ret, 1 << 20)
    rt = R.rope_table(N, R.inv_freq(H.D, base, dev))
    run = lambda s: interface._flash_attn_fwd(q[s].to(dev), k[s].to(dev), v[s].to(dev), atflash_window_zhi=zhi,  # noqa: E731
                                              rope=rt)
    out, lse = run(slice(0, B))
    for b in range(B):
        o1, l1 = run(slice(b, b + 1))
        assert torch.equal(out[b], o1[0]) and torch.equal(lse[b], l1[0]), f"sequence {b}"
    ref = H.prefill_oracle(q[B - 1:], k[B - 1:], v[B - 1:], base, k_ret, rope=True)
    H.assert_close(out[B - 1:], ref, "last sequence")
