"""Ragged decode (kf_attn_decode_ragged_kernel): decode with key counts whose
waves share the stages that the sequences really hold.

Shapes where the division can go wrong: empty sequences and single keys, one
long sequence among short ones (a head over many workers), hundreds of heads
inside one worker's share, more than 64 and 192 sequences (the batch map's
registers), more than 256 and 4096 (its blocks, of 64 and 128), counts past the capacity, 1 to 16 rows per KV head (both ways of
merging), every head dimension, page sizes from 16 rows, invalid page ids.
Bar as in the other parity tests (fp64 oracle), and the same call by the
capacity's splits (a workspace of only those partials) within 2e-4:
P is rounded to fp16 against other row maxima, 2^-11 of values of order 1.
"""
import numpy as np
import pytest

import kernelfoundry_amd as kf
from oracle import attn_oracle as orc
from tests._parity import capacity_workspace, run_and_check


def _lens(kind, B, cap, seed):
    rng = np.random.default_rng(seed)
    if kind == "one_long":
        n = rng.integers(0, 40, B)
        n[B // 2] = cap
    elif kind == "short":
        n = rng.integers(1, 70, B)
    elif kind == "full":
        n = np.full(B, cap)
    elif kind == "empty":
        n = np.zeros(B)
    else:
        n = np.exp(rng.uniform(np.log(cap / 16), np.log(cap), B))
        n[:3] = (0, 1, cap + 9)  # none, one key, clamped
    return n.astype(np.int32)


CASES = [
    # B, H_q, H_kv, q_len, cap, D, page_size (0: contiguous), lengths, causal
    (16, 32, 8, 1, 4096, 128, 0, "mixed", False),
    (16, 32, 8, 4, 4096, 128, 0, "mixed", True),       # 16 rows: merged in LDS
    (32, 32, 8, 1, 8192, 128, 16, "one_long", False),
    (70, 8, 8, 2, 2048, 128, 64, "mixed", True),       # > 64 sequences
    (130, 8, 4, 1, 1024, 128, 32, "short", False),
    (16, 32, 8, 1, 4096, 128, 16, "full", False),
    (16, 32, 8, 1, 4096, 128, 16, "empty", False),
    (24, 16, 16, 1, 2048, 64, 128, "mixed", False),
    (20, 32, 4, 2, 3000, 64, 0, "one_long", True),     # 16 rows, ragged capacity
    (64, 16, 16, 1, 4000, 16, 0, "mixed", False),
    (96, 4, 2, 3, 4096, 16, 16, "one_long", True),
    (16, 16, 4, 1, 4096, 256, 16, "mixed", False),
    (16, 16, 4, 3, 4096, 256, 0, "one_long", True),    # 12 rows
    (256, 8, 2, 1, 512, 128, 16, "mixed", False),      # the registers' last sequence
    (257, 8, 2, 1, 512, 128, 0, "mixed", False),       # one block more than them
    (700, 4, 2, 3, 300, 64, 0, "one_long", True),
    (1000, 16, 4, 1, 200, 256, 0, "short", False),
    (4500, 4, 2, 1, 64, 16, 16, "short", False),       # blocks of 128 sequences
    (4500, 4, 2, 1, 64, 16, 0, "one_long", False),
]


def _id(c):
    return "B{}_Hq{}_Hkv{}_q{}_cap{}_D{}_ps{}_{}".format(*c[:8])


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_cases_take_the_ragged_kernel(case):
    B, H_q, H_kv, q, cap, D, ps, kind, causal = case
    cap = -(-cap // ps) * ps if ps else cap
    names = kf.kernel_names(B, q, cap, H_q, H_kv, D, causal=causal, masked=True)
    assert names == f"kf_attn_decode_ragged_kernel<{D}, false> + kf_attn_ragged_merge_kernel<{D}>"
    assert kf.workspace_bytes_lens(B, q, cap, H_q, H_kv, D) >= kf.workspace_bytes(B, q, cap, H_q, H_kv, D)
    if ps:
        assert kf.paged_workspace_bytes(B, q, H_q, H_kv, D, ps, cap // ps) == \
            kf.workspace_bytes_lens(B, q, cap, H_q, H_kv, D)


def test_other_calls_keep_their_kernels_and_workspace():
    # Equal lengths take it where the split grid is several rounds of
    # workgroups (96 heads, not 64 or 128), and are asked for its workspace.
    assert "ragged" in kf.kernel_names(12, 1, 4096, 32, 8, 128)
    assert kf.workspace_bytes(12, 1, 4096, 32, 8, 128) == kf.workspace_bytes_lens(12, 1, 4096, 32, 8, 128)
    for B in (8, 16, 32):
        assert "ragged" not in kf.kernel_names(B, 1, 4096, 32, 8, 128)
    # Small capacities and more than 16 rows per KV head never; larger ones for
    # eight rows and more, and at D = 16, unless there is a head per worker.
    for shape in ((2048, 1, 128, 8, 1, 128), (4096, 1, 64, 4, 2, 16)):
        assert "ragged" in kf.kernel_names(*shape, masked=True)
    for shape in ((4, 1, 4096, 32, 8, 128), (1, 1, 4096, 32, 8, 128), (64, 1, 4096, 32, 1, 64),
                  (256, 1, 1024, 8, 1, 128), (64, 1, 4096, 8, 1, 128), (298, 1, 336, 16, 2, 64),
                  (361, 1, 368, 4, 2, 16), (9, 1, 31616, 8, 1, 64), (28, 4, 1984, 24, 8, 128)):
        assert "ragged" not in kf.kernel_names(*shape, masked=True)
        assert kf.workspace_bytes_lens(*shape) == kf.workspace_bytes(*shape)
    # A workspace of the capacity's plan is enough (the call then ends at
    # its first HIP call on a host without a GPU), one byte less is not.
    import torch
    if torch.cuda.is_available():
        return
    fake, ws = 1 << 20, 1 << 24
    for B in (16, 32):
        need = kf.workspace_bytes(B, 1, 4096, 32, 8, 128)
        for flags in (0, kf.KF_ATTN_LSE):
            def call(n, w=ws):
                return kf.attn_fwd_ex_ptr(fake, fake, fake, fake, 0, 0, B, 1, 4096, 32, 8, 128,
                                          kv_lens=fake, flags=flags, workspace=w, workspace_bytes=n)
            assert call(need) == kf.KF_ERR_HIP
            assert call(kf.workspace_bytes_lens(B, 1, 4096, 32, 8, 128)) == kf.KF_ERR_HIP
            if need:
                assert call(need - 1) == kf.KF_ERR_WORKSPACE
                assert call(need, ws + 16) == kf.KF_ERR_ALIGN
            else:
                assert call(0, 0) == kf.KF_ERR_HIP


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_ragged_parity(case):
    import torch
    B, H_q, H_kv, q, cap, D, ps, kind, causal = case
    cap = -(-cap // ps) * ps if ps else cap
    print("case", case, flush=True)
    lens = _lens(kind, B, cap, 11 + B)
    rng = np.random.default_rng(B + D)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    q16 = rng.standard_normal((B, H_q, q, D), dtype=np.float32).astype(np.float16)
    Q, L = dev(q16), dev(lens)
    used = np.minimum(lens, cap)
    if ps:
        need = -(-used // ps)
        pool = int(need.sum()) + 5
        kp, vp = (rng.standard_normal((pool, H_kv, ps, D), dtype=np.float32).astype(np.float16)
                  for _ in range(2))
        table = np.full((B, cap // ps), -1, dtype=np.int32)
        ids, at = rng.permutation(pool), 0
        for b in range(B):
            table[b, :need[b]] = ids[at:at + need[b]]
            at += need[b]
        for b in rng.integers(0, B, 3):      # pages that do not exist
            if need[b] > 1:
                table[b, rng.integers(0, need[b])] = pool + 3
        K, V, T = dev(kp), dev(vp), dev(table)
        O, Mi, Li = kf.attn_decode_paged(Q, K, V, T, L, return_stats=True, causal=causal)
        O16, lse = kf.attn_decode_paged(Q, K, V, T, L, out_dtype=torch.float16, return_lse=True,
                                        causal=causal)
        kc, valid = orc.paged_to_contiguous(kp, table, ps)
        vc, _ = orc.paged_to_contiguous(vp, table, ps)
        by_capacity = kf.attn_decode_paged(Q, K, V, T, L, causal=causal,
                                           workspace=capacity_workspace(B, q, cap, H_q, H_kv, D))
    else:
        kc, vc = (rng.standard_normal((B, H_kv, cap, D), dtype=np.float32).astype(np.float16)
                  for _ in range(2))
        K, V, valid = dev(kc), dev(vc), None
        O, Mi, Li = kf.attn_fwd(Q, K, V, return_stats=True, causal=causal, kv_lens=L)
        O16, lse = kf.attn_fwd(Q, K, V, out_dtype=torch.float16, return_lse=True, causal=causal, kv_lens=L)
        # The same by the capacity's splits.
        n = kf.workspace_bytes(B, q, cap, H_q, H_kv, D)
        ws = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
        by_capacity = torch.empty_like(O)
        st = kf.attn_fwd_ex_ptr(Q.data_ptr(), K.data_ptr(), V.data_ptr(), by_capacity.data_ptr(), 0, 0, B, q,
                                cap, H_q, H_kv, D, kv_lens=L.data_ptr(),
                                flags=kf.KF_ATTN_CAUSAL if causal else 0, workspace=ws.data_ptr(),
                                workspace_bytes=n, stream=torch.cuda.current_stream().cuda_stream)
        assert st == kf.KF_OK
    torch.cuda.synchronize()
    Or, Mr, Lr = orc.sdpa(q16, kc, vc, causal=causal, kv_lens=[int(x) for x in used],
                          **({"key_valid": valid} if valid is not None else {}))
    assert (O - by_capacity).abs().max().item() <= 2e-4 * max(1.0, np.abs(Or).max())
    O, Mi, Li, lse = (x.cpu().numpy() for x in (O, Mi, Li, lse))
    assert np.isfinite(O).all()
    empty = np.isneginf(Mr)
    assert np.array_equal(np.isneginf(Mi), empty) and np.array_equal(np.isneginf(lse), empty)
    assert (O[empty] == 0).all() and (Li[empty] == 0).all()
    full = ~empty
    if full.any():
        ok, max_abs, rel = orc.within_tolerance(O, Or)
        assert ok, f"max_abs={max_abs:.3g} rel={rel:.3g}"
        assert np.abs(Mi[full] - Mr[full]).max() <= 1e-4
        assert np.abs(Li[full] / Lr[full] - 1).max() <= 1e-3
        assert np.abs(lse[full] - (Mr[full] + np.log(Lr[full]))).max() <= 1e-3
    # The same rows, rounded once.
    assert np.array_equal(O16.cpu().numpy(), O.astype(np.float16))


# Without key counts: equal lengths that end inside a stage, both ways of
# merging, every head dimension.
EVEN = [
    # B, H_q, H_kv, q_len, kv_len, D, causal
    (132, 8, 4, 2, 4078, 16, True),
    (108, 8, 4, 1, 1258, 16, False),
    (25, 16, 16, 1, 777, 64, False),
    (60, 16, 16, 2, 1487, 64, True),
    (12, 32, 8, 1, 4099, 128, False),
    (21, 16, 4, 2, 1001, 256, True),
]


def _even_id(c):
    return "B{}_Hq{}_Hkv{}_q{}_kv{}_D{}".format(*c[:6])


@pytest.mark.parametrize("case", EVEN, ids=_even_id)
def test_equal_lengths_take_the_ragged_kernel(case):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: the plan is for its CU count")
    B, H_q, H_kv, q, kv, D, causal = case
    names = kf.kernel_names(B, q, kv, H_q, H_kv, D, causal=causal)
    assert names == f"kf_attn_decode_ragged_kernel<{D}, false> + kf_attn_ragged_merge_kernel<{D}>"
    # At D = 16 only grids of many rounds.
    assert "ragged" not in kf.kernel_names(19, 1, 12123, 4, 2, 16)


@pytest.mark.gpu
@pytest.mark.parametrize("case", EVEN, ids=_even_id)
def test_equal_lengths_parity(case):
    B, H_q, H_kv, q, kv, D, causal = case
    run_and_check(B, H_q, H_kv, q, kv, D, causal, None, seed=900 + B)


@pytest.mark.gpu
def test_ragged_decode_replayed_with_other_key_counts():
    """One captured call, replayed several times with other key counts in the
    same array and eager work between: every replay has the bits of an eager
    call with those counts (the division is found on the device)."""
    import torch
    B, q, cap, H_q, H_kv, D = 16, 1, 4096, 32, 8, 128
    print("case replay", flush=True)
    assert "ragged" in kf.kernel_names(B, q, cap, H_q, H_kv, D, masked=True)
    normal = lambda *s: torch.randn(s, device="cuda", dtype=torch.float16)
    Q, K, V = normal(B, H_q, q, D), normal(B, H_kv, cap, D), normal(B, H_kv, cap, D)
    lens = torch.full((B,), cap, dtype=torch.int32, device="cuda")
    ws = torch.empty(kf.workspace_bytes_lens(B, q, cap, H_q, H_kv, D), dtype=torch.uint8, device="cuda")
    out = torch.empty((B, H_q, q, D), dtype=torch.float32, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        kf.attn_fwd(Q, K, V, out, kv_lens=lens, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        kf.attn_fwd(Q, K, V, out, kv_lens=lens, workspace=ws)
    for kind in ("mixed", "full", "empty", "one_long", "short", "mixed"):
        lens.copy_(torch.from_numpy(_lens(kind, B, cap, 3)))
        ref = kf.attn_fwd(Q, K, V, kv_lens=lens)
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), kind


@pytest.mark.gpu
@pytest.mark.parametrize("B,q,ps", [(16, 1, 16), (16, 4, 16), (12, 1, 0), (16, 4, 0)])
def test_ragged_infinity_and_nan(B, q, ps):
    """An infinity in a sequence's last V row, in a stage that other rows do
    not fill, stays one and does not become NaN (0 times it; paged calls:
    contiguous ones repeat that row), a query row of NaN gives NaN and no
    other row does.  (The build does not honour NaNs, so that is what this
    compiler makes of the merges and no promise.)  q = 1 and 4: partials straight to memory and by LDS."""
    import torch
    H_q, H_kv, cap, D = 32, 8, 4096, 128
    print("case", B, q, ps, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B + q)
    normal = lambda *s: torch.randn(s, generator=gen, device="cuda", dtype=torch.float16)
    lens = torch.tensor([1001 + 61 * b for b in range(B)], dtype=torch.int32, device="cuda")
    Q = normal(B, H_q, q, D)
    Q[1, 5, q - 1] = float("nan")
    if ps:
        need = cap // ps
        K, V = normal(B * need, H_kv, ps, D), normal(B * need, H_kv, ps, D)
        T = torch.arange(B * need, dtype=torch.int32, device="cuda").view(B, need)
        last = int(lens[0]) - 1
        V[T[0, last // ps].long(), :, last % ps, 7] = float("inf")
        O = kf.attn_decode_paged(Q, K, V, T, lens)
        assert torch.isposinf(O[0, :, :, 7]).all()
        O[0, :, :, 7] = 0
    else:
        K, V = normal(B, H_kv, cap, D), normal(B, H_kv, cap, D)
        O = kf.attn_fwd(Q, K, V, kv_lens=lens)
    assert torch.isnan(O[1, 5, q - 1]).all()
    O[1, 5, q - 1] = 0
    assert torch.isfinite(O).all()


@pytest.mark.gpu
def test_noalloc_takes_no_scratch_where_the_plan_needs_none():
    """kf_attn_fwd_noalloc shares its scratch between all calls on a device: a
    call whose capacity plan is unsplit stays on that plan, so that it may run
    next to another.  Bit for bit the call without a workspace."""
    import torch
    lib = kf.load_library()
    B, q, cap, H_q, H_kv, D = shape = (32, 1, 4096, 32, 8, 128)
    assert kf.workspace_bytes(*shape) == 0 < kf.workspace_bytes_lens(*shape)
    print("case", shape, flush=True)
    normal = lambda *s: torch.randn(s, device="cuda", dtype=torch.float16)
    Q, K, V = normal(B, H_q, q, D), normal(B, H_kv, cap, D), normal(B, H_kv, cap, D)
    lens = torch.from_numpy(_lens("mixed", B, cap, 5)).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    A, C = torch.empty_like(Q, dtype=torch.float32), torch.empty_like(Q, dtype=torch.float32)
    assert lib.kf_attn_fwd_noalloc(Q.data_ptr(), K.data_ptr(), V.data_ptr(), A.data_ptr(), None, None, *shape,
                                   lens.data_ptr(), 0, stream) == kf.KF_OK
    assert kf.attn_fwd_ex_ptr(Q.data_ptr(), K.data_ptr(), V.data_ptr(), C.data_ptr(), 0, 0, *shape,
                              kv_lens=lens.data_ptr(), stream=stream) == kf.KF_OK
    torch.cuda.synchronize()
    assert torch.equal(A, C)
