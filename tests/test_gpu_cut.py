"""GPU parity of the cut passes (cut_hist_kernel and the launches after it)
against the oracle, bit-exact: rows that keep many tokens by top-p, a large
top-k or a low min-p floor. The cases sit where the passes can go wrong: bins
that hold one token, every token, or more than the chunk lists and the LDS list
take (ties, constant rows, a range far off); boundaries in the first and the
last bin; vocabularies of one chunk, of one token past a chunk, and whole rows;
temperatures that leave one weight or all weights; rows of infinities and NaN;
masks, stops and penalties; drafts with kept and unkept tokens."""
import numpy as np
import pytest

import jf_sampler as J
from jf_sampler import workloads as WL
from harness import NO, assert_same, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def check(V, pols, **kw):
    print(f"case V={V} rows={len(pols)} keys={sorted(kw)}", flush=True)
    g, r = run_gpu(V, pols, **kw), run_oracle(V, pols, **kw)
    assert_same(g, r)
    return g


def policies(V):
    return [J.policy(temperature=0.8, top_p=0.95), J.policy(temperature=1.0, top_p=0.5),
            J.policy(temperature=0.05, top_p=0.9), J.policy(temperature=30.0, top_p=0.999),
            J.policy(temperature=1.0, top_p=1e-6), J.policy(temperature=1.0, top_p=0.9999999),
            J.policy(temperature=1.0, top_k=max(1, min(1025, V - 1))),
            J.policy(temperature=0.9, top_k=max(1, V // 2), top_p=0.9),
            J.policy(temperature=2.0, top_k=max(1, V - 1), top_p=0.3),
            J.policy(temperature=3.0, min_p=0.001), J.policy(temperature=2.0, min_p=0.01, top_p=0.8),
            J.policy(temperature=1.5, min_p=0.002, top_k=max(1, min(3000, V - 1)), top_p=0.97)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V", [1100, 8192, 8193, 3 * 8192 + 5, 70001, 151936])
def test_cut_rows(V, bf16):
    rng = np.random.default_rng(V + bf16)
    pols = policies(V)
    x = rng.normal(0, 2.5, (len(pols), V)).astype(np.float32)
    u = rng.random(len(pols)).astype(np.float32)
    u[:3] = 0.0, np.float32(1.0 - 2.0 ** -24), 0.5
    kw = dict(logits_bf16=WL.to_bf16_bits(x)) if bf16 else dict(logits=x)
    check(V, pols, uniforms=u, kept_capacity=V if V < 20000 else 5000, **kw)


@pytest.mark.parametrize("decimals", [0, 1, 2])
def test_cut_ties(decimals):
    """Rounded values: the boundary bin holds from hundreds to tens of
    thousands of tied tokens, past the chunk lists (1008) and the LDS list
    (3072)."""
    V = 60001
    rng = np.random.default_rng(decimals)
    pols = policies(V)
    x = np.round(rng.normal(0, 2.0, (len(pols), V)), decimals).astype(np.float32)
    check(V, pols, logits=x, uniforms=rng.random(len(pols)).astype(np.float32),
          kept_capacity=4000)


def test_cut_extreme_rows():
    """Constant rows, one value above all, values past the bins' range, and
    rows of infinities, NaN and the lowest finite value."""
    V = 20001
    rng = np.random.default_rng(3)
    low = np.float32(-3.402823466e38)
    rows = []
    for fill in (0.0, -0.0, 5.0, low, -np.inf, np.nan, np.inf):
        rows.append(np.full(V, fill, np.float32))
    one = np.full(V, -50.0, np.float32)
    one[777] = 3.0
    rows.append(one)
    far = rng.normal(0, 1, V).astype(np.float32)
    far[::3] = -1e9
    far[1::5] = -np.inf
    rows.append(far)
    wide = (rng.normal(0, 1, V) * 1e4).astype(np.float32)
    rows.append(wide)
    signs = np.zeros(V, np.float32)
    signs[::2] = -0.0
    rows.append(signs)
    nans = rng.normal(0, 2, V).astype(np.float32)
    nans[rng.random(V) < 0.9] = np.nan
    rows.append(nans)
    x = np.stack(rows)
    for p in (J.policy(temperature=0.8, top_p=0.95), J.policy(temperature=1.0, top_k=1500),
              J.policy(temperature=1.0, top_k=15000, top_p=0.7),
              J.policy(temperature=1.0, min_p=1e-6, top_p=0.9)):
        check(V, [p] * len(rows), logits=x, uniforms=rng.random(len(rows)).astype(np.float32),
              kept_capacity=3000)


@pytest.mark.parametrize("dense", [False, True])
def test_cut_drafted(dense):
    """Drafted rows: the draft's token kept, unkept or outside the row; a q
    that takes everything (the plain draw) and one that takes nothing."""
    V = 30011
    rng = np.random.default_rng(17 + dense)
    base = [J.policy(temperature=0.8, top_p=0.95), J.policy(temperature=1.0, top_k=2000),
            J.policy(temperature=1.0, top_k=4000, top_p=0.9),
            J.policy(temperature=2.0, min_p=0.003)]
    pols = [base[i % 4] for i in range(16)]
    x = rng.normal(0, 2.0, (16, V)).astype(np.float32)
    best = x.argmax(1)
    draft = np.where(np.arange(16) % 4 < 2, best, rng.integers(0, V, 16)).astype(np.uint32)
    draft[3], draft[5] = NO, np.uint32(x[5].argmin())
    kw = dict(draft_tokens=draft, drafted_rows=14)
    if dense:
        q = rng.dirichlet(np.ones(V) * 0.05, 16).astype(np.float32)
        q[1] = 1.0
        q[2] = 0.0
        kw["dense_q"] = q
    else:
        cid = rng.integers(0, V, (16, 16)).astype(np.uint32)
        cid[:, 0] = draft
        kw.update(cand_ids=cid, cand_probs=rng.dirichlet(np.ones(16), 16).astype(np.float32))
    check(V, pols, logits=x, uniforms=rng.random(16).astype(np.float32), **kw)
    check(V, pols, logits=x, uniforms=rng.random(16).astype(np.float32), kept_capacity=700, **kw)


def test_cut_masks_penalties_and_other_rows():
    """Masked rows (from 1 admitted token up), stop exclusion and penalties,
    among greedy, listed and uncut rows of one call; repeated on one sampler,
    so words an earlier call left must not matter."""
    V = 50003
    rng = np.random.default_rng(23)
    pols, hist = [], []
    allowed = rng.random((18, V)) < 0.02
    allowed[0] = False
    allowed[0, 4242] = True
    for r in range(18):
        kw = [dict(temperature=0.8, top_p=0.9, constrained=True),
              dict(temperature=1.0, top_k=1500, repetition=1.2, presence=0.4),
              dict(), dict(temperature=0.7, top_k=40), dict(temperature=1.0),
              dict(temperature=1.2, top_p=0.97, frequency=0.3, exclude_stop=True)][r % 6]
        pols.append(J.policy(**kw))
        pen = "presence" in kw or "frequency" in kw
        hist.append(rng.integers(0, V, 700).astype(np.uint32) if pen else None)
    x = rng.normal(0, 2.5, (18, V)).astype(np.float32)
    stop = (int(x[5].argmax()), int(x[11].argmax()))
    s = J.Sampler(V, 18)
    kw = dict(logits=x, masks=WL.mask_words(allowed), stop=stop, histories=hist,
              generated=[350 if h is not None else 0 for h in hist], mark_prompt=[True] * 18)
    for _ in range(3):
        check(V, pols, uniforms=rng.random(18).astype(np.float32), sampler=s, **kw)
        check(V, pols[::-1], uniforms=rng.random(18).astype(np.float32), sampler=s,
              **{**kw, "histories": hist[::-1], "generated": kw["generated"][::-1]})
    plain = [J.policy(temperature=1.0)] * 18  # the self-validating words' launch, after
    check(V, plain, logits=x, uniforms=rng.random(18).astype(np.float32), sampler=s)
    s.close()


def test_cut_rows_past_a_grid_dimension():
    """More rows than a grid has blocks in y: the cut passes' kept outputs of
    every 997th row and of the last ones, and every greedy row among them."""
    import torch
    V, rows = 128, 65600
    rng = np.random.default_rng(31)
    x = rng.normal(0, 2.5, (rows, V)).astype(np.float32)
    u = rng.random(rows).astype(np.float32)
    kinds = [J.policy(temperature=0.8, top_p=0.9), J.policy(),
             J.policy(temperature=1.0, top_k=100, top_p=0.95)]
    pols = [kinds[r % 3] for r in range(rows)]
    some = sorted(set(range(0, rows, 997)) | set(range(32766, 32772)) |
                  set(range(65533, 65540)) | set(range(rows - 4, rows)))
    print(f"case rows={rows}", flush=True)
    g = run_gpu(V, pols, logits=x, uniforms=u, kept_capacity=V)
    pick = {k: v[some] for k, v in g.items()}
    assert_same(pick, run_oracle(V, [pols[r] for r in some], logits=x[some], uniforms=u[some],
                                 kept_capacity=V))
    np.testing.assert_array_equal(g["tokens"][1::3], x[1::3].argmax(1))
    assert (g["tokens"] < V).all() and (g["kept_counts"][0::3] > 0).all()
    torch.cuda.empty_cache()
