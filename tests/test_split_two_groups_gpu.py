"""Split prefill on the two-KV-group layout (128 rows per workgroup): partitions
that end inside a tile, rows that end inside a row tile, groups and partitions
past a sequence's keys, rows that see no key, a workspace for fewer partitions.
"""
import pytest

import kernelfoundry_amd as kf
from tests._parity import run_and_check

CASES = [
    # B, H_q, H_kv, q_len, kv_len, D, causal, kv_lens
    (1, 32, 8, 128, 8192, 128, True, None),
    (1, 16, 4, 300, 6001, 128, False, None),             # ragged rows and keys
    (1, 32, 4, 500, 4095, 128, True, None),              # unsplit by the four-group layout
    (2, 16, 4, 256, 5000, 64, True, [5000, 130]),        # partitions past 130 keys, rows without any
    (2, 16, 4, 256, 5000, 64, False, [0, 4999]),         # an empty sequence
    (1, 32, 8, 243, 9605, 128, True, [1300]),            # keys shared by all partitions
    (3, 8, 2, 256, 9000, 128, False, [1, 65, 1111]),     # partitions of one tile, and without keys
]


def _name(c):
    return kf.kernel_names(c[0], c[3], c[4], c[1], c[2], c[5], causal=c[6], masked=c[7] is not None)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}_q{}_kv{}_D{}".format(c[0], *c[3:6]))
def test_plans(case):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: the plan is for its CU count")
    B, H_q, H_kv, q, kv, D, causal, lens = case
    p = kf.plan(B, q, kv, H_q, H_kv, D)
    assert p.path == "prefill_split" and p.kv_per_split % 64 == 0
    mask = "true" if causal or lens else "false"
    assert _name(case).startswith(f"kf_attn_prefill_kernel<{D}, {mask}, 8, 2> + kf_attn_split_merge_kernel<{D}, ")
    assert p.grid_blocks == B * H_kv * -(-(H_q // H_kv * q) // 128) * p.num_splits <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}_q{}_kv{}_D{}".format(c[0], *c[3:6]))
def test_parity(case):
    run_and_check(*case, seed=700 + case[3])


@pytest.mark.gpu
def test_smaller_workspaces_agree():
    """Workspaces for all, two and no partitions: the same O to 2e-4 (P is
    rounded to fp16 against other row maxima)."""
    import torch
    B, H_q, H_kv, q, kv, D = 1, 32, 8, 256, 8192, 128
    print("case smaller workspaces", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    Q, K, V = (torch.randn((B, h, n, D), generator=g, dtype=torch.float16, device="cuda")
               for h, n in ((H_q, q), (H_kv, kv), (H_kv, kv)))
    ref = kf.attn_fwd(Q, K, V, causal=True)
    full = kf.workspace_bytes(B, q, kv, H_q, H_kv, D)
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    for n in (full, full * 2 // kf.plan(B, q, kv, H_q, H_kv, D).num_splits, 0):
        O = torch.full_like(ref, float("nan"))
        st = kf.attn_fwd_ex_ptr(Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), 0, 0, B, q, kv, H_q,
                                H_kv, D, flags=kf.KF_ATTN_CAUSAL, workspace=ws.data_ptr() if n else 0,
                                workspace_bytes=n, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert st == kf.KF_OK and (O - ref).abs().max().item() <= 2e-4


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_partitions_share_a_short_sequences_keys(D):
    """Every partition of a sequence that fills an eighth of its capacity has
    keys (a finite row maximum in its partials), one that fills all of it gives
    the bits of the call without key counts."""
    import torch
    B, H_q, H_kv, q, kv = 1, 32, 8, 256, 8192
    print("case short sequence", D, flush=True)
    p = kf.plan(B, q, kv, H_q, H_kv, D)
    assert p.path == "prefill_split" and "8, 2>" in kf.kernel_names(B, q, kv, H_q, H_kv, D, masked=True)
    g = torch.Generator(device="cuda").manual_seed(9)
    Q, K, V = (torch.randn((B, h, n, D), generator=g, dtype=torch.float16, device="cuda")
               for h, n in ((H_q, q), (H_kv, kv), (H_kv, kv)))
    ws = torch.zeros(p.workspace_bytes // 4, dtype=torch.float32, device="cuda")
    lens = lambda n: torch.tensor([n], dtype=torch.int32, device="cuda")
    kf.attn_fwd(Q, K, V, kv_lens=lens(kv // 8), workspace=ws)
    parts = p.num_splits * B * H_q * q           # O partials, then the row maxima
    assert torch.isfinite(ws[parts * D:parts * (D + 1)]).all()
    assert torch.equal(kf.attn_fwd(Q, K, V, kv_lens=lens(kv)), kf.attn_fwd(Q, K, V, kv_lens=None))


@pytest.mark.parametrize("shape,layout", [
    # B, q_len, kv_len, H_q, H_kv; us in four groups (split or not), in two
    ((1, 256, 1024, 32, 8), "8, 4>"),        # 11.8, 13.4
    ((6, 64, 2048, 32, 8), "8, 4>"),         # 19.3, 22.2
    ((2, 149, 1741, 32, 1), "8, 4>"),        # 15.9, 17.1
    ((2, 256, 4096, 32, 8), "8, 4>"),        # 32.5, 34.3
    ((1, 256, 8192, 32, 8), "8, 2> + kf_attn_split_merge"),   # 36.1, 31.9
    ((4, 128, 8192, 16, 16), "8, 2> + kf_attn_split_merge"),  # 51.2, 37.1
])
def test_d64_takes_the_faster_layout(shape, layout):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: the plan is for its CU count")
    assert f"kf_attn_prefill_kernel<64, true, {layout}" in kf.kernel_names(*shape, 64, causal=True)
