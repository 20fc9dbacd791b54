"""Unsplit causal prefill layouts of their own: two KV groups inside the 8-wave
kernel (one round of 256-row tiles), 4-wave workgroups (tiles that straddle
heads, short prompts), the 128-row KV-group kernel at D = 256; and the order
and placement of causal row tiles where q_len is no multiple of the tile and
where KV heads share XCDs (1, 2, 3, 4, 12 heads).

Every query row of every head must be written once, by the right tile: whole
outputs are compared with a float64 softmax on the GPU, to the parity bar (max
2e-3, rel L2 1e-2), Mi to 1e-4 and Li to 1e-3 relative.
"""
import pytest

import kernelfoundry_amd as kf

PREFILL = "kf_attn_prefill_kernel<{}, true, {}, {}>"
WIDE = "kf_attn_prefill_wide_kernel<{}, true, {}, {}>"
CASES = [
    # B, H_q, H_kv, q_len, kv_len, D, kernel
    (1, 32, 8, 2048, 2048, 128, PREFILL.format(128, 8, 1)),   # two groups inside
    (1, 32, 8, 2048, 2600, 128, PREFILL.format(128, 8, 1)),   # the same, kv_len > q_len
    (1, 32, 1, 2048, 2048, 64, PREFILL.format(64, 8, 1)),     # the same, one KV head on 8 XCDs
    (1, 32, 8, 2200, 2200, 128, PREFILL.format(128, 4, 1)),   # tiles straddle heads
    (3, 32, 4, 1000, 1011, 128, PREFILL.format(128, 4, 1)),   # 12 KV heads: 4 sets of 3
    (4, 32, 8, 1024, 1024, 128, PREFILL.format(128, 4, 1)),   # short, two rounds
    (3, 32, 4, 1000, 1000, 64, PREFILL.format(64, 4, 2)),
    (3, 64, 1, 700, 700, 64, PREFILL.format(64, 4, 2)),       # 3 KV heads on 8 XCDs
    (2, 16, 4, 1500, 1500, 256, WIDE.format(256, 2, "false")),
    (1, 16, 2, 1300, 1400, 256, WIDE.format(256, 2, "false")),
    (4, 32, 8, 1024, 700, 128, PREFILL.format(128, 8, 1)),    # fewer keys than queries: as before
    (2, 32, 1, 300, 300, 128, PREFILL.format(128, 4, 2)),     # 2 KV heads, 64-row tiles, ragged
    (3, 2, 1, 5000, 5000, 64, PREFILL.format(64, 8, 4)),      # long rows, 3 heads
    # One query head per KV head, 12 of them (4 sets of 3, side by side) and 36
    # (4 sets of 9, the plain placement).
    (1, 12, 12, 5900, 5900, 128, PREFILL.format(128, 8, 1)),
    (3, 12, 12, 2048, 2048, 128, PREFILL.format(128, 8, 1)),
    # D = 64: full rounds of 256-row tiles, tiles that do not straddle, tiles that pad.
    (8, 16, 16, 400, 400, 64, PREFILL.format(64, 8, 1)),
    (16, 32, 1, 256, 256, 64, PREFILL.format(64, 8, 1)),
    (8, 16, 16, 700, 700, 64, PREFILL.format(64, 4, 2)),
    (9, 16, 16, 1024, 1024, 64, PREFILL.format(64, 4, 2)),
    (11, 16, 16, 713, 713, 64, PREFILL.format(64, 8, 1)),
]


def _id(c):
    return "B{}_Hq{}_Hkv{}_q{}_kv{}_D{}".format(*c[:6])


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_kernels(case):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: the plan is for its CU count")
    B, H_q, H_kv, q, kv, D, name = case
    assert kf.kernel_names(B, q, kv, H_q, H_kv, D, causal=True) == name


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [False, True], ids=["full", "lens"])
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_parity(case, lens):
    import torch
    B, H_q, H_kv, q, kv, D, _ = case
    print("case", case, lens, flush=True)
    g = torch.Generator(device="cuda").manual_seed(q + D)
    Q, K, V = (torch.randn((B, h, n, D), generator=g, dtype=torch.float16, device="cuda")
               for h, n in ((H_q, q), (H_kv, kv), (H_kv, kv)))
    # Key counts below kv_len, the last below q_len (rows without keys).
    counts = [max(kv - 37 * (b + 1), 5) if b < B - 1 else min(kv, q) // 3 for b in range(B)] if lens else [kv] * B
    L = torch.tensor(counts, dtype=torch.int32, device="cuda") if lens else None
    O, Mi, Li = kf.attn_fwd(Q, K, V, causal=True, kv_lens=L, return_stats=True)
    ratio = H_q // H_kv
    keys = torch.arange(kv, device="cuda")
    for b in range(B):
        limit = (torch.arange(q, device="cuda") + counts[b] - q + 1).clamp(0, counts[b])
        for h in range(H_q):
            k, v = K[b, h // ratio].double(), V[b, h // ratio].double()
            s = Q[b, h].double() @ k.t().contiguous() / D ** 0.5
            s = s.masked_fill(keys >= limit[:, None], float("-inf"))
            seen = limit > 0
            m = s.max(dim=1).values
            p = torch.exp(s - torch.where(seen, m, torch.zeros_like(m))[:, None])
            l = p.sum(dim=1)
            ref = torch.where(seen[:, None], p @ v / l[:, None], torch.zeros((), dtype=torch.float64, device="cuda"))
            err = O[b, h].double() - ref
            assert torch.isfinite(O[b, h]).all()
            assert err.abs().max() <= 2e-3 and err.norm() <= 1e-2 * ref.norm(), (b, h, err.abs().max().item())
            assert torch.equal(Mi[b, h].isneginf(), ~seen) and (Li[b, h][~seen] == 0).all()
            assert (Mi[b, h].double() - m)[seen].abs().max() <= 1e-4
            assert (Li[b, h].double() / l - 1)[seen].abs().max() <= 1e-3
