"""GPU parity of kf_attn_decode_paged (decode over a paged K/V cache).

The pools, block tables and query are seeded; the oracle gathers the pages
into per-sequence K/V (oracle.paged_to_contiguous, pinned against the
reference's own torch gather) and runs the fp64 sdpa with the sequences' key
counts, causal mask and page validity.  Bar: max |got - ref| <= 2e-3 and
||got - ref||_2 / ||ref||_2 <= 1e-2 for O, Mi to 1e-4, Li to 1e-3 relative,
empty rows exactly O = 0, Mi = -inf, Li = 0.

Cases: page sizes 16 (two pages per 32-row stage) to 256, random page
permutations (the reference's worst-case fragmentation), GQA / MQA / MHA,
q_len 1 and small causal q_len, every head dimension, ragged and empty
sequences, invalid page ids inside a sequence, on both decode kernels (the
short-split kernel's paged form for small jobs, the streaming kernel for
large ones); and bitwise equality with the contiguous decode of either
kernel when the pages hold the same rows in order.
"""
import numpy as np
import pytest

from oracle import attn_oracle as orc
from tests._parity import capacity_workspace

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need the MI355X"
    return torch


def _announce(**kw):
    print("case", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


def _paged_inputs(B, H_q, H_kv, q_len, D, page_size, max_pages, num_pages, kv_lens, seed,
                  bad_ids=()):
    rng = np.random.default_rng(seed)
    f16 = lambda a: a.astype(np.float32).astype(np.float16)
    q16 = f16(rng.standard_normal((B, H_q, q_len, D)))
    k16 = f16(rng.standard_normal((num_pages, H_kv, page_size, D)))
    v16 = f16(rng.standard_normal((num_pages, H_kv, page_size, D)))
    perm = rng.permutation(num_pages)
    table = np.full((B, max_pages), -1, dtype=np.int32)
    used = 0
    for b in range(B):
        n = min(max_pages, (kv_lens[b] + page_size - 1) // page_size)
        table[b, :n] = perm[used:used + n]
        used += n
    for b, pg, val in bad_ids:
        table[b, pg] = val
    return q16, k16, v16, table, np.asarray(kv_lens, dtype=np.int32)


def _oracle(q16, k16, v16, table, lens, page_size, causal):
    K, valid = orc.paged_to_contiguous(k16, table, page_size)
    V, _ = orc.paged_to_contiguous(v16, table, page_size)
    return orc.sdpa(q16, K, V, causal=causal, kv_lens=lens, key_valid=valid)


def _run(q16, k16, v16, table, lens, causal, by_capacity=False):
    import kernelfoundry_amd as kf
    torch = _torch()
    ws = None
    if by_capacity:
        B, H_q, q_len, D = q16.shape
        ws = capacity_workspace(B, q_len, k16.shape[2] * table.shape[1], H_q, k16.shape[1], D)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    O, Mi, Li = kf.attn_decode_paged(t(q16), t(k16), t(v16), t(table), t(lens),
                                     return_stats=True, causal=causal, workspace=ws)
    torch.cuda.synchronize()
    return O.cpu().numpy(), Mi.cpu().numpy(), Li.cpu().numpy()


def _check(got, ref, label):
    O, Mi, Li = got
    Or, Mr, Lr = ref
    assert np.isfinite(O).all(), f"{label}: non-finite O"
    ok, max_abs, rel = orc.within_tolerance(O, Or)
    assert ok, f"{label}: max_abs={max_abs:.3g} rel={rel:.3g}"
    empty = np.isneginf(Mr)
    assert np.array_equal(np.isneginf(Mi), empty), f"{label}: Mi = -inf on the wrong rows"
    assert (O[empty] == 0).all() and (Li[empty] == 0).all(), f"{label}: empty rows not zero"
    full = ~empty
    if full.any():
        assert np.abs(Mi[full] - Mr[full]).max() <= 1e-4, f"{label}: Mi"
        rel_l = np.abs(Li[full] - Lr[full]).max() / np.abs(Lr[full]).max()
        assert rel_l <= 1e-3, f"{label}: Li rel err {rel_l:.3g}"


PAGED_CASES = [
    # B, H_q, H_kv, q_len, D, page_size, max_pages, kv_lens, causal, bad_ids
    (2, 32, 8, 1, 128, 16, 70, [1100, 517], False, ()),
    (3, 32, 8, 1, 128, 32, 40, [1280, 1, 0], False, ()),
    (2, 16, 2, 2, 64, 64, 20, [1200, 700], True, ()),
    (1, 32, 1, 1, 64, 256, 9, [2048], False, ()),            # MQA, C4b-like
    (2, 8, 8, 1, 16, 16, 30, [477, 33], False, ()),           # MHA, D=16
    (2, 8, 2, 4, 256, 32, 12, [350, 200], True, ()),          # D=256, causal q_len=4
    (2, 32, 8, 1, 128, 16, 64, [1024, 1000], False, [(0, 3, -5), (1, 10, 10 ** 6)]),
    (4, 32, 4, 1, 128, 128, 33, [4200, 3000, 129, 4224], False, ()),
    # Jobs large enough for the ragged decode, and given a workspace of the
    # plan's partials for the streaming decode kernel, with invalid page ids
    # (the ones above run the short-split kernel's paged form, the last of them
    # the streaming kernel's).
    (12, 32, 8, 1, 128, 16, 256, [4096 - 53 * b for b in range(12)], False,
     [(0, 3, -5), (5, 200, 10 ** 6)]),
    (24, 16, 16, 1, 64, 64, 40, [2560 - 100 * b for b in range(24)], False, [(7, 0, -1)]),
    (12, 32, 8, 2, 256, 32, 64, [2048 - 77 * b for b in range(12)], True, [(11, 9, -2)]),
]


def test_paged_cases_reach_both_decode_kernels():
    """The cases above run the paged forms of the short-split kernel and, as
    they are and by the capacity's splits, of the ragged and the streaming
    decode at D = 64, 128 and 256, with invalid page ids (the planner sizes a
    paged decode like a contiguous one over the capacity)."""
    import kernelfoundry_amd as kf
    kinds = set()
    for B, H_q, H_kv, q_len, D, ps, max_pages, kv_lens, causal, bad in PAGED_CASES:
        shape = B, q_len, ps * max_pages, H_q, H_kv, D
        name = kf.kernel_names(*shape, causal=causal, masked=True).split("<")[0]
        stream = kf.plan(*shape).splits_per_block == 1    # the plan's own kernel
        assert stream == (name != "kf_attn_decode_short_kernel")
        kinds.add((name, D if "ragged" in name else 0, bool(bad)))
    assert kinds >= {("kf_attn_decode_short_kernel", 0, True), ("kf_attn_decode_short_kernel", 0, False),
                     ("kf_attn_decode_kernel", 0, False)}
    assert kinds >= {("kf_attn_decode_ragged_kernel", D, True) for D in (64, 128, 256)}


@pytest.mark.parametrize("case", PAGED_CASES, ids=lambda c: "B{}_Hq{}_Hkv{}_q{}_D{}_ps{}_{}{}".format(
    c[0], c[1], c[2], c[3], c[4], c[5], "causal" if c[8] else "full", "_bad" if c[9] else ""))
def test_paged_decode_parity(case):
    B, H_q, H_kv, q_len, D, ps, max_pages, kv_lens, causal, bad = case
    num_pages = B * max_pages + 7
    _announce(test="paged", B=B, H_q=H_q, H_kv=H_kv, q_len=q_len, D=D, page_size=ps,
              max_pages=max_pages, kv_lens=kv_lens, causal=causal, bad=bad)
    q16, k16, v16, table, lens = _paged_inputs(B, H_q, H_kv, q_len, D, ps, max_pages, num_pages,
                                               kv_lens, 900 + D + ps, bad)
    ref = _oracle(q16, k16, v16, table, lens, ps, causal)
    for by_capacity in (False, True):
        got = _run(q16, k16, v16, table, lens, causal, by_capacity)
        _check(got, ref, f"case {case} by_capacity={by_capacity}")


@pytest.mark.parametrize("page_size", [16, 32, 64])
def test_paged_short_split_in_order_equals_contiguous_bitwise(page_size):
    """The configs[1] decode (B = 1, 32 / 8 heads, 4096 keys) over pages that
    hold a contiguous cache's rows in order: the short-split kernel's paged
    form computes exactly what its contiguous form computes (same splits,
    same loads, same arithmetic), O, Mi and Li bit for bit, also with a key
    count that ends inside a page."""
    import kernelfoundry_amd as kf
    torch = _torch()
    B, H_q, H_kv, D, max_pages = 1, 32, 8, 128, 4096 // page_size
    cap = max_pages * page_size
    assert kf.plan(B, 1, cap, H_q, H_kv, D).splits_per_block == 4   # short-split kernel
    q16, k16, v16 = orc.normal_fp16_inputs(B, H_q, H_kv, 1, cap, D, 2718)
    to_pages = lambda a: a.reshape(B, H_kv, max_pages, page_size, D).transpose(0, 2, 1, 3, 4) \
        .reshape(B * max_pages, H_kv, page_size, D)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    # Pages in a shuffled pool, the table pointing at them in order.
    perm = np.random.default_rng(page_size).permutation(B * max_pages).astype(np.int32)
    kp, vp = np.empty_like(to_pages(k16)), np.empty_like(to_pages(v16))
    kp[perm], vp[perm] = to_pages(k16), to_pages(v16)
    table = perm.reshape(B, max_pages)
    for klen in (cap, cap - 7):
        _announce(test="paged_short_vs_contiguous", page_size=page_size, kv_len=klen)
        lens = np.array([klen], dtype=np.int32)
        Op, Mp, Lp = kf.attn_decode_paged(t(q16), t(kp), t(vp), t(table), t(lens), return_stats=True)
        Oc, Mc, Lc = kf.attn_fwd(t(q16), t(k16), t(v16), kv_lens=t(lens), return_stats=True)
        torch.cuda.synchronize()
        assert torch.equal(Op, Oc) and torch.equal(Mp, Mc) and torch.equal(Lp, Lc)


@pytest.mark.parametrize("page_size", [16, 64])
def test_paged_in_order_equals_contiguous_bitwise(page_size):
    """Pages holding the rows of a contiguous cache in order: the paged kernel
    computes exactly what kf_attn_fwd_ex computes on the contiguous cache
    (same splits, same stages, same arithmetic): the ragged decode on both,
    and given a workspace of the plan's partials the streaming decode."""
    import kernelfoundry_amd as kf
    torch = _torch()
    B, H_q, H_kv, D, max_pages = 12, 32, 8, 128, 4096 // page_size
    cap = max_pages * page_size
    assert kf.plan(B, 1, cap, H_q, H_kv, D).splits_per_block == 1
    assert "decode_ragged" in kf.kernel_names(B, 1, cap, H_q, H_kv, D, masked=True)
    _announce(test="paged_vs_contiguous", page_size=page_size)
    q16, k16, v16 = orc.normal_fp16_inputs(B, H_q, H_kv, 1, cap, D, 314)
    to_pages = lambda a: a.reshape(B, H_kv, max_pages, page_size, D).transpose(0, 2, 1, 3, 4) \
        .reshape(B * max_pages, H_kv, page_size, D)
    table = np.arange(B * max_pages, dtype=np.int32).reshape(B, max_pages)
    lens = np.array([cap - 37 * b for b in range(B)], dtype=np.int32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    outs = []
    for ws in (None, capacity_workspace(B, 1, cap, H_q, H_kv, D)):
        Op = kf.attn_decode_paged(t(q16), t(to_pages(k16)), t(to_pages(v16)), t(table), t(lens), workspace=ws)
        Oc = kf.attn_fwd(t(q16), t(k16), t(v16), kv_lens=t(lens), workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(Op, Oc)
        outs.append(Oc)
    assert not torch.equal(*outs)   # two kernels
