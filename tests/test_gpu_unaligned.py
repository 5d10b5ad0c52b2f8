"""Rows that start at any element: every kernel that reads logits (or a dense
draft q) 16 bytes a lane, on views whose rows start 1..7 elements past a
16-byte boundary with odd strides, against the oracle, bit-exact. The
vocabularies end inside a vector, on one and past one, so the last loads'
clamps are at the edge of the row; the rows before and after hold values that
would win if a load strayed."""
import numpy as np
import pytest

import jf_sampler as J
from jf_sampler import workloads as WL
from harness import run_oracle

pytestmark = pytest.mark.gpu
NO = 0xFFFFFFFF


def view(host, offset, gap, fill):
    """A device view of `host` [rows][V] whose rows start `offset` elements
    into a buffer of V + gap elements a row, every other element `fill`."""
    import torch
    rows, V = host.shape
    buf = torch.full((offset + rows * (V + gap) + 16,), fill, dtype=host.dtype, device="cuda")
    out = buf[offset:offset + rows * (V + gap)].view(rows, V + gap)[:, :V]
    out.copy_(host)
    return out


KINDS = {
    "greedy": (dict(repetition=1.2), dict()),
    "uncut": (dict(temperature=1.0), dict(temperature=0.7)),
    "listed": (dict(temperature=0.7, top_k=50, top_p=0.9), dict(temperature=1.0, min_p=0.1)),
    "cut": (dict(temperature=0.8, top_p=0.95), dict(temperature=1.0, top_k=1500)),
}


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("kind", list(KINDS) + ["mixed", "drafted"])
@pytest.mark.parametrize("V,offset,gap", [(8191, 1, 0), (16385, 3, 2), (24580, 2, 1),
                                          (8200, 5, 7), (9, 1, 0)])
def test_rows_at_any_element(kind, bf16, V, offset, gap):
    import torch
    rng = np.random.default_rng(V + offset)
    rows = 8
    print(f"case {kind} bf16={bf16} V={V} offset={offset} gap={gap}", flush=True)
    both = [p for k in KINDS.values() for p in k] if kind == "mixed" else \
        list(KINDS["uncut"]) + list(KINDS["listed"]) if kind == "drafted" else list(KINDS[kind])
    kws = [dict(both[r % len(both)]) for r in range(rows)]
    for k in kws:
        if k.get("top_k", 0) >= V:
            k["top_k"] = V // 2
    pols = [J.policy(**k) for k in kws]
    x = rng.normal(0, 2.5, (rows, V)).astype(np.float32)
    bits = WL.to_bf16_bits(x)
    host = torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16) if bf16 else \
        torch.from_numpy(x)
    lg = view(host, offset, gap, 1000.0)
    u = rng.random(rows).astype(np.float32)
    hist = [rng.integers(0, V, 40).astype(np.uint32) if "repetition" in k else None for k in kws]
    kw, ref = {}, {}
    table = J.PenaltyTable(V, rows, 64)
    for r, h in enumerate(hist):
        if h is not None:
            table.rebuild(r, h, 20, None, True)
    if kind == "drafted":
        draft = rng.integers(0, V, rows).astype(np.uint32)
        draft[1], draft[2] = x[1].argmax(), x[2].argmax()
        q = rng.dirichlet(np.ones(V) * 0.05, rows).astype(np.float32)
        dq = view(torch.from_numpy(q), offset, gap, 7.0)
        kw = dict(draft_tokens=torch.from_numpy(draft.view(np.int32)).cuda(), dense_q=dq)
        ref = dict(draft_tokens=draft, dense_q=q)
    out = torch.zeros(rows, dtype=torch.int32, device="cuda")
    dp = torch.zeros(rows, dtype=torch.float32, device="cuda")
    s = J.Sampler(V, rows)
    s.sample(lg, pols, out, uniforms=torch.from_numpy(u).cuda(), penalties=table,
             penalty_rows=list(range(rows)), out_draft_probs=dp, **kw)
    torch.cuda.synchronize()
    want = run_oracle(V, pols, histories=hist, generated=[20] * rows, mark_prompt=[True] * rows,
                      uniforms=u, **(dict(logits_bf16=bits) if bf16 else dict(logits=x)), **ref)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), want["tokens"])
    if kind == "drafted":
        np.testing.assert_array_equal(dp.cpu().numpy(), want["draft_probs"])
    s.close()
    table.close()


@pytest.mark.parametrize("V,offset", [(8193, 1), (20003, 3)])
def test_draft_rows_at_any_element(V, offset):
    """The draft selector's top 16 of rows past a 16-byte boundary, by value
    and lowest id."""
    import torch
    print(f"case draft V={V} offset={offset}", flush=True)
    rng = np.random.default_rng(V)
    lanes = 2
    x = np.round(rng.normal(0, 2.0, (lanes * 8, V)), 2).astype(np.float32)
    lg = view(torch.from_numpy(x), offset, 1, 1000.0)
    z = torch.zeros
    cand = z((lanes * 7, 16), dtype=torch.int32, device="cuda")
    unary = z((lanes * 7, 16), dtype=torch.float32, device="cuda")
    tokens = z(lanes * 7, dtype=torch.int32, device="cuda")
    book = z((V, 256), dtype=torch.int16, device="cuda")
    s = J.DraftSelector(V, lanes)
    s.launch(s.args(logits=lg, hidden=z((lanes * 8, 256), dtype=torch.int16, device="cuda"),
                    pred_codebook=book, succ_codebook=book, anchors=[1, 2],
                    policies=[J.policy()] * lanes, candidates=cand, unary=unary, tokens=tokens,
                    stride=lg.stride(0)))
    torch.cuda.synchronize()
    for l in range(lanes):
        for p in range(7):
            row = x[l * 8 + p + 1]
            want = np.lexsort((np.arange(V), -row))[:16]
            np.testing.assert_array_equal(cand.cpu().numpy()[l * 7 + p], want)
            np.testing.assert_array_equal(unary.cpu().numpy()[l * 7 + p], row[want])
    s.close()
