"""Batches with greedy rows whose entries name no uniform of theirs: the greedy
rows' tokens, and their neighbours' draws, against the oracle through every
launch that finishes such a batch (the small and the general merge, the uncut
draw, the cut passes' last launch, the residual launch). The entries point at a
slot of NaN (inside the buffer: which address a kernel may read is checked on
the host, tests/test_launch_plan.py)."""
import numpy as np
import pytest

import jf_sampler as J
from harness import NO, run_oracle

pytestmark = pytest.mark.gpu

ROW = {"g": dict(), "k": dict(temperature=0.7, top_k=50, top_p=0.9),
       "n": dict(temperature=0.8, top_p=0.95), "u": dict(temperature=1.0),
       "d": dict(temperature=1.0), "m": dict(temperature=1.0, min_p=0.05)}


@pytest.mark.parametrize("indexed", [True, False])
@pytest.mark.parametrize("kinds", ["kgkgk", "gmg", "gugug", "gnkug", "ng", "dgugd", "kgd"])
def test_greedy_rows_without_uniforms(kinds, indexed):
    import torch
    V, rows = 20003, len(kinds)
    print(f"case {kinds} indexed={indexed}", flush=True)
    rng = np.random.default_rng(rows + indexed)
    pols = [J.policy(**ROW[k]) for k in kinds]
    x = rng.normal(0, 2.5, (rows, V)).astype(np.float32)
    u = rng.random(rows).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    kw, ref = {}, {}
    if "d" in kinds:
        draft = np.array([x[r].argmax() if k == "d" else NO for r, k in enumerate(kinds)],
                         np.uint32)
        q = rng.dirichlet(np.ones(V) * 0.05, rows).astype(np.float32)
        kw = dict(draft_tokens=dev(draft.view(np.int32)), dense_q=dev(q),
                  draft_token_index=[r if k == "d" else NO for r, k in enumerate(kinds)])
        ref = dict(draft_tokens=draft, dense_q=q)
    if indexed:
        # The sampled rows' uniforms in any order, a slot of NaN at the end.
        place = rng.permutation(rows)
        buf = np.full(rows + 1, np.nan, np.float32)
        buf[place] = u
        index = np.where([k == "g" for k in kinds], rows, place).astype(np.int32)
        kw["uniform_index"] = dev(index)
    else:
        buf = np.where([k == "g" for k in kinds], np.float32(np.nan), u).astype(np.float32)
    out = torch.zeros(rows, dtype=torch.int32, device="cuda")
    s = J.Sampler(V, rows)
    keep = s.sample(dev(x), pols, out, uniforms=dev(buf), **kw)
    torch.cuda.synchronize()
    del keep
    want = run_oracle(V, pols, logits=x, uniforms=u, **ref)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), want["tokens"])
    s.close()
