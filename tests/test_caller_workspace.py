"""The caller's workspace in the Python entries: used whenever the call runs
with it, refused only where the call cannot do without one and the buffer is
no workspace (another device, not contiguous)."""
import numpy as np
import pytest

import kernelfoundry_amd as kf

# (B, q_len, kv_len, H_q, H_kv, D): bytes of the partials of the plan that needs
# least, O and the two statistics.
LEAST = [
    ((16, 1, 4096, 32, 8, 128), 2),    # split decode, two splits
    ((32, 1, 4096, 32, 8, 128), 0),    # unsplit decode
    ((1, 256, 8192, 32, 8, 128), 2),   # split prefill, four-group layout: two partitions
    ((1, 512, 16384, 32, 8, 128), 0),  # prefill that only the two-group layout splits
    ((1, 512, 512, 32, 8, 128), 0),
]


@pytest.mark.parametrize("shape,splits", LEAST, ids=lambda v: str(v))
def test_least_workspace(shape, splits):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: the plan is for its CU count")
    B, q, _, H_q, _, D = shape
    up = lambda n: -(-n // 256) * 256
    parts = splits * B * H_q * q
    assert kf.workspace_bytes_least(*shape) == up(4 * parts * D) + 2 * up(4 * parts)
    assert kf.workspace_bytes_least(*shape) <= kf.workspace_bytes(*shape) <= kf.workspace_bytes_lens(*shape)
    assert kf.workspace_bytes_least(1, 1, 1, 3, 2, 128) == 0   # invalid


def test_plan_describes_the_call_given_its_partials():
    """kf_attn_plan and kf_attn_kernel_names: a decode that is named by the
    ragged decode is described by the splits it runs with less workspace, all
    others by the plan's own kernel and the workspace it asks for."""
    rng = np.random.default_rng(5)
    up = lambda n: -(-n // 256) * 256
    seen = set()
    for _ in range(400):
        D = int(rng.choice([16, 64, 128, 256]))
        H_kv = int(rng.choice([1, 2, 4, 8, 16]))
        H_q = H_kv * int(rng.choice([1, 2, 4, 8]))
        shape = B, q, kv, *_ = (int(2 ** rng.uniform(0, 8)), int(rng.integers(1, 5)), int(2 ** rng.uniform(5, 15)),
                                H_q, H_kv, D)
        p = kf.plan(*shape)
        least = kf.workspace_bytes_least(*shape)
        parts = p.num_splits * B * H_q * q if p.num_splits > 1 else 0
        assert p.workspace_bytes == kf.workspace_bytes(*shape) >= least
        if p.path not in ("decode", "decode_split"):
            continue
        assert least == up(4 * parts * D) + 2 * up(4 * parts)
        ragged = "decode_ragged" in kf.kernel_names(*shape)
        assert ragged or p.workspace_bytes == least
        assert not ragged or (p.path == "decode_split" and p.splits_per_block == 1)
        assert ("decode_short" in kf.kernel_names(*shape)) == (p.splits_per_block == 4)
        seen.add((ragged, p.path))
    assert {(True, "decode_split"), (False, "decode_split"), (False, "decode")} <= seen


def test_the_callers_buffer_is_taken_where_the_call_runs_with_it():
    import torch
    cpu = torch.device("cpu")

    def ws(n, need, least):
        mine = torch.empty(n, dtype=torch.uint8)
        got, size = kf._workspace(torch, mine, need, lambda: least, cpu, None)
        return ("mine" if got is mine else "new" if got is not None else None), size

    assert ws(64, 0, 0) == (None, 0)
    assert ws(64, 64, 32) == ("mine", 64) and ws(100, 64, 32) == ("mine", 64)
    assert ws(63, 64, 32) == ("mine", 63) and ws(32, 64, 32) == ("mine", 32)   # by a smaller plan
    assert ws(31, 64, 32) == ("new", 64)
    assert ws(0, 64, 0) == ("mine", 0)
    assert kf._workspace(torch, None, 64, None, cpu, None)[1] == 64


def test_a_buffer_that_is_no_workspace():
    import torch
    meta = torch.empty(4096, dtype=torch.uint8, device="meta")     # another device
    strided = torch.empty(4096, dtype=torch.uint8)[::2]
    cpu = torch.device("cpu")
    for bad in (meta, strided):
        with pytest.raises(ValueError):
            kf._workspace(torch, bad, 64, lambda: 32, cpu, None)
        got, size = kf._workspace(torch, bad, 64, lambda: 0, cpu, None)
        assert got is not bad and got.device == cpu and size == 64


@pytest.mark.gpu
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B", [16, 32])
def test_entries_use_a_workspace_of_the_capacity_plan(B, paged):
    """A workspace of the plan's own bytes runs the capacity's splits (the bits
    of the C ABI given as much), one of the best size the ragged decode."""
    import torch
    shape = (B, 1, 4096, 32, 8, 128)
    H_q, H_kv, cap, D, ps = 32, 8, 4096, 128, 64
    print("case", shape, paged, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B)
    normal = lambda *s: torch.randn(s, generator=gen, dtype=torch.float16, device="cuda")
    Q = normal(B, H_q, 1, D)
    lens = torch.tensor([1 + 127 * b for b in range(B)], dtype=torch.int32, device="cuda")
    K, V = normal(B, H_kv, cap, D), normal(B, H_kv, cap, D)
    least = kf.workspace_bytes_least(*shape)
    assert (least > 0) == (B == 16)
    small = torch.empty(least, dtype=torch.uint8, device="cuda")
    other = torch.empty(1 << 20, dtype=torch.uint8)                # host memory
    ref = torch.empty_like(Q, dtype=torch.float32)
    given = dict(workspace=small.data_ptr(), workspace_bytes=least,
                 stream=torch.cuda.current_stream().cuda_stream)
    if paged:
        pages = lambda x: x.view(B, H_kv, cap // ps, ps, D).transpose(1, 2).reshape(-1, H_kv, ps, D).contiguous()
        table = torch.arange(B * cap // ps, dtype=torch.int32, device="cuda").view(B, -1)
        Kp, Vp = pages(K), pages(V)
        run = lambda ws: kf.attn_decode_paged(Q, Kp, Vp, table, lens, workspace=ws)
        st = kf.attn_decode_paged_ptr(Q.data_ptr(), Kp.data_ptr(), Vp.data_ptr(), table.data_ptr(), lens.data_ptr(),
                                      ref.data_ptr(), 0, 0, B, 1, H_q, H_kv, D, ps, cap // ps, Kp.shape[0], **given)
    else:
        run = lambda ws: kf.attn_fwd(Q, K, V, kv_lens=lens, workspace=ws)
        st = kf.attn_fwd_ex_ptr(Q.data_ptr(), K.data_ptr(), V.data_ptr(), ref.data_ptr(), 0, 0, *shape,
                                kv_lens=lens.data_ptr(), **given)
    assert st == kf.KF_OK
    best = run(None)
    assert torch.equal(run(small), ref) and not torch.equal(best, ref)
    assert (best - ref).abs().max().item() <= 2e-4
    assert torch.equal(run(torch.empty(kf.workspace_bytes_lens(*shape), dtype=torch.uint8, device="cuda")), best)
    if least:
        with pytest.raises(ValueError):
            run(other)
    else:
        assert torch.equal(run(other), best)
