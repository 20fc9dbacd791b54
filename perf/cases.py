"""The attention calls that programs make of this library, as cases to time.

A case names one call of a public entry point: ``attn_fwd`` on torch tensors
(entry "torch"), the raw-pointer form of the C ABI with a workspace that the
program keeps ("c"), or decode over a paged cache (paged).  The listed cases
are the ordinary work of a serving or training program over its range of
sizes; ``draw`` gives more calls of the same kinds.

Fields of a case: B, q_len, kv_len (rows allocated per head; of a paged cache
its capacity), H_q, H_kv, D, causal, out ("f32" / "f16" / "bf16"), lse,
lens_seed (-1: every sequence has kv_len keys; else the draw of the
sequences' key counts), page_size (0: contiguous), entry.
"""
import random

import torch

import kernelfoundry_amd as kf

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FLAGS = {"f32": 0, "f16": kf.KF_ATTN_OUT_F16, "bf16": kf.KF_ATTN_OUT_BF16}
# H_q, H_kv, D: GQA as in the repository's bench, its MQA row, its D = 256
# rows, D = 64 GQA, and multi-head attention as encoders have it.
HEADS = ((32, 8, 128), (32, 8, 128), (32, 8, 128), (32, 1, 64), (16, 4, 256), (32, 8, 64),
         (16, 16, 64), (32, 1, 128), (8, 8, 128), (4, 2, 16))


def _case(name, B, q_len, kv_len, heads=(32, 8, 128), causal=False, out="f32", lse=False,
          lens_seed=-1, page_size=0, entry="torch"):
    H_q, H_kv, D = heads
    c = {"B": B, "q_len": q_len, "kv_len": kv_len, "H_q": H_q, "H_kv": H_kv, "D": D,
         "causal": causal, "out": out, "lse": lse, "lens_seed": lens_seed,
         "page_size": page_size, "entry": entry}
    return dict(c, name=name) if name else c


def listed():
    return [
        # One token of one sequence, MQA: the smallest call, all latency.
        _case("decode_mqa_b1", 1, 1, 2048, heads=(32, 1, 64), entry="c"),
        # One token of one sequence with GQA and a 4096-token context.
        _case("decode_b1", 1, 1, 4096, entry="c"),
        # A full batch of equally long contexts: the HBM-bound decode.
        _case("decode_b32", 32, 1, 8192),
        # Speculative verification: 4 tokens a sequence, over a pre-allocated
        # cache that the sequences fill to different lengths.
        _case("verify_ragged_b16", 16, 4, 4096, causal=True, out="f16", lens_seed=3),
        # A serving step: one token for each sequence of a batch over a paged
        # cache, contexts of very different lengths.
        _case("paged_ragged_b32", 32, 1, 8192, out="f16", lens_seed=1, page_size=16, entry="c"),
        # Prompts: short, middling, long.  Language models mask causally.
        _case("prefill_causal_512", 1, 512, 512, causal=True, out="f16"),
        _case("prefill_causal_2048", 1, 2048, 2048, causal=True, out="f16"),
        _case("prefill_causal_8192", 1, 8192, 8192, causal=True, out="f16", lse=True),
        # The repository's headline: S = 4096, unmasked, fp32 out.
        _case("prefill_4096", 1, 4096, 4096),
        # Chunked prefill: 256 new tokens against a long context.
        _case("chunk_256x8192", 1, 256, 8192, causal=True, out="f16"),
        # An encoder's padded batch: multi-head, odd length, key counts.
        _case("encoder_padded_b8", 8, 1000, 1000, heads=(16, 16, 64), out="f16", lens_seed=2),
        # D = 256, two odd-length prompts.
        _case("prefill_d256_1500", 2, 1500, 1500, heads=(16, 4, 256), causal=True, out="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    most = [work(c) for c in listed()]
    flops, nbytes = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    while True:
        H_q, H_kv, D = heads = rng.choice(HEADS)
        kind = rng.choice(("decode", "ragged", "paged", "paged", "prefill", "prefill", "chunk",
                           "encoder"))
        kw = {"out": rng.choice(("f32", "f16", "f16", "bf16")), "lse": rng.random() < 0.2,
              "entry": rng.choice(("torch", "c"))}
        seed = rng.randrange(1 << 20)
        if kind in ("decode", "ragged", "paged"):
            q_len = rng.choice([n for n in (1, 1, 1, 2, 4) if H_q // H_kv * n <= 32])
            B, kv = _log(rng, 1, 64), _log(rng, 256, 16384)
            if kind == "ragged":
                kw["entry"] = "torch"
            if kind == "paged":
                page = rng.choice((16, 16, 32, 64, 128))
                kv = -(-kv // page) * page
                kw["page_size"] = page
            c = _case("", B, q_len, kv, heads, causal=q_len > 1,
                      lens_seed=-1 if kind == "decode" else seed, **kw)
        elif kind == "prefill":
            S = _log(rng, 64, 8192)
            S = S if rng.random() < 0.5 else -(-S // 64) * 64
            c = _case("", _log(rng, 1, 8), S, S, heads, causal=rng.random() < 0.75, **kw)
        elif kind == "chunk":
            c = _case("", _log(rng, 1, 8), _log(rng, 16, 512), _log(rng, 1024, 16384), heads,
                      causal=True, lens_seed=-1 if rng.random() < 0.6 else seed, **kw)
        else:
            S = _log(rng, 64, 2048)
            c = _case("", _log(rng, 2, 32), S, S, heads, lens_seed=seed, **kw)
        w = work(c)
        if w["flops"] <= flops and w["bytes"] <= nbytes:
            return c


def _lens(case):
    """The sequences' key counts: spread over a factor of 16 below the
    capacity, many short ones and few long ones."""
    if case["lens_seed"] < 0:
        return [case["kv_len"]] * case["B"]
    r, top = random.Random(case["lens_seed"]), case["kv_len"]
    least = min(case["q_len"], top) if case["causal"] else 1
    return [max(least, _log(r, max(1.0, top / 16), top)) for _ in range(case["B"])]


def work(case):
    B, q, H_q, H_kv, D = (case[k] for k in ("B", "q_len", "H_q", "H_kv", "D"))
    pairs = keys = 0
    for n in _lens(case):
        keys += n
        # Causal, aligned to the last key: query i sees keys j <= i + n - q.
        lo = max(n - q + 1, 0)
        pairs += (lo + n) * (n - lo + 1) // 2 if case["causal"] else q * n
    rows = B * H_q * q
    nbytes = rows * D * (2 + (4 if case["out"] == "f32" else 2)) + keys * H_kv * D * 4
    nbytes += rows * 4 if case["lse"] else 0
    if case["page_size"]:
        nbytes += 4 * sum(-(-n // case["page_size"]) for n in _lens(case))
    return {"bytes": nbytes, "flops": 4 * pairs * H_q * D}


def _inputs(case, seed):
    """Q, K, V (page pools of a paged cache), key counts and block table."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=gen, dtype=torch.float16, device=dev)

    B, q, kv, H_q, H_kv, D = (case[k] for k in ("B", "q_len", "kv_len", "H_q", "H_kv", "D"))
    order = random.Random(seed)
    lens = _lens(case)
    order.shuffle(lens)
    Q = normal(B, H_q, q, D)
    counts = table = None
    if case["lens_seed"] >= 0 or case["page_size"]:
        counts = torch.tensor(lens, dtype=torch.int32, device=dev)
    if case["page_size"]:
        # Pages placed at random in a pool with some pages to spare.
        page = case["page_size"]
        need = [-(-n // page) for n in lens]
        pool = sum(need) + sum(need) // 16 + 1
        ids = list(range(pool))
        order.shuffle(ids)
        rows = []
        for n in need:
            rows.append(ids[:n] + [0] * (-(-kv // page) - n))
            ids = ids[n:]
        table = torch.tensor(rows, dtype=torch.int32, device=dev)
        K, V = normal(pool, H_kv, page, D), normal(pool, H_kv, page, D)
    else:
        K, V = normal(B, H_kv, kv, D), normal(B, H_kv, kv, D)
    return Q, K, V, counts, table, lens


def prepare(case, seed):
    Q, K, V, counts, table, _ = _inputs(case, seed)
    s = {"case": case, "Q": Q, "K": K, "V": V, "counts": counts, "table": table}
    # A decode loop writes each step's output to the same buffer.
    B, q, kv, H_q, H_kv, D = (case[k] for k in ("B", "q_len", "kv_len", "H_q", "H_kv", "D"))
    if case["entry"] == "c":
        s["out"] = torch.empty_like(Q, dtype=DTYPES[case["out"]])
        s["lse"] = torch.empty((B, H_q, q), dtype=torch.float32, device=Q.device) if case["lse"] else None
        if case["page_size"]:
            need = kf.paged_workspace_bytes(B, q, H_q, H_kv, D, case["page_size"], table.shape[1])
        else:
            need = kf.workspace_bytes(B, q, kv, H_q, H_kv, D)
        s["ws"] = torch.empty(max(need, 256), dtype=torch.uint8, device=Q.device)
        s["need"] = need
        s["stream"] = torch.cuda.current_stream().cuda_stream
        s["flags"] = (FLAGS[case["out"]] | (kf.KF_ATTN_CAUSAL if case["causal"] else 0)
                      | (kf.KF_ATTN_LSE if case["lse"] else 0))
    return s


def run(s):
    c = s["case"]
    if c["entry"] == "torch":
        kw = {"causal": c["causal"], "kv_lens": s["counts"], "out_dtype": DTYPES[c["out"]],
              "return_lse": c["lse"]}
        if c["page_size"]:
            return kf.attn_decode_paged(s["Q"], s["K"], s["V"], s["table"], kw.pop("kv_lens"), **kw)
        return kf.attn_fwd(s["Q"], s["K"], s["V"], **kw)
    Q, K, V, out, lse, ws = s["Q"], s["K"], s["V"], s["out"], s["lse"], s["ws"]
    counts = s["counts"].data_ptr() if s["counts"] is not None else 0
    lse_ptr = lse.data_ptr() if lse is not None else 0
    if c["page_size"]:
        st = kf.attn_decode_paged_ptr(
            Q.data_ptr(), K.data_ptr(), V.data_ptr(), s["table"].data_ptr(), counts,
            out.data_ptr(), lse_ptr, 0, c["B"], c["q_len"], c["H_q"], c["H_kv"], c["D"],
            c["page_size"], s["table"].shape[1], K.shape[0], flags=s["flags"],
            workspace=ws.data_ptr(), workspace_bytes=s["need"], stream=s["stream"])
    else:
        st = kf.attn_fwd_ex_ptr(
            Q.data_ptr(), K.data_ptr(), V.data_ptr(), out.data_ptr(), lse_ptr, 0, c["B"],
            c["q_len"], c["kv_len"], c["H_q"], c["H_kv"], c["D"], kv_lens=counts,
            flags=s["flags"], workspace=ws.data_ptr(), workspace_bytes=s["need"],
            stream=s["stream"])
    if st != kf.KF_OK:
        raise kf.KfError(st, kf.status_string(st))
    return (out, lse) if lse is not None else out


def tolerance(case):
    """Four times the error against float64 that was measured over the listed
    cases and two dozen drawn ones: rel 1.3e-4 - 2.9e-4 with fp32 or fp16 out
    (P is rounded to fp16), 1.7e-3 with bf16 out; the largest value 7.8e-3
    off (causal, the rows that see few keys)."""
    return {"rel": 7e-3 if case["out"] == "bf16" else 1.2e-3, "max": 3e-2}


def exact(case, seed):
    """softmax(Q K^T / sqrt(D)) V in float64, one KV head and a block of its
    query rows at a time."""
    Q, K, V, _, table, lens = _inputs(case, seed)
    B, q, H_q, H_kv, D = (case[k] for k in ("B", "q_len", "H_q", "H_kv", "D"))
    ratio = H_q // H_kv
    out = torch.empty(Q.shape, dtype=torch.float64, device=Q.device)
    lse = torch.empty(Q.shape[:3], dtype=torch.float64, device=Q.device)
    for b in range(B):
        n = lens[b]
        if case["page_size"]:
            pages = table[b, : -(-n // case["page_size"])].long()
        # Query row r of a KV head (all its query heads together) is query r % q.
        limit = torch.arange(q, device=Q.device).repeat(ratio) + (n - q + 1)
        for h in range(H_kv):
            if case["page_size"]:
                k, v = (x[pages, h].reshape(-1, D)[:n].double() for x in (K, V))
            else:
                k, v = K[b, h, :n].double(), V[b, h, :n].double()
            kt = k.t().contiguous()
            rows = Q[b, h * ratio : (h + 1) * ratio].reshape(-1, D).double()
            o = out[b, h * ratio : (h + 1) * ratio].view(-1, D)
            e = lse[b, h * ratio : (h + 1) * ratio].view(-1)
            step = max(1, (1 << 26) // n)
            for r in range(0, rows.shape[0], step):
                s = rows[r : r + step] @ kt / D ** 0.5
                if case["causal"]:
                    s.masked_fill_(torch.arange(n, device=Q.device) >= limit[r : r + step, None],
                                   float("-inf"))
                e[r : r + step] = torch.logsumexp(s, dim=1)
                o[r : r + step] = torch.exp(s - e[r : r + step, None]) @ v
    return (out, lse) if case["lse"] else out
