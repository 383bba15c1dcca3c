"""GPU parity of the prefill kernel's balanced grid: the call's key steps in equal runs, one per block, and a merge of
the tiles that a run boundary cuts.

The planner takes it where a block per 128-row tile leaves CUs idle or waits for the longest sequence.  Cases at the
places where the runs can go wrong: boundaries inside, at and between tiles; tiles over more than 8 and more than 64
runs; fewer steps than CUs; causal limits that leave a run without keys (fresh prompts); more than 64 sequences (the
device scan's second round) with decodes among them; hints that do not match the device tables; token pages; one-group
blocks (head_dim > 128).  Every output row must be written and meet 1e-5 (F32) / 2e-3 (F16) against the oracle.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mvr_attn as M  # noqa: E402
import oracle as O  # noqa: E402
import workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-5, "f16": 2e-3}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M.load_library()
    O.build()


# dtype, query heads, KV heads, head_dim, page size, new tokens, cached tokens, hints
CASES = {
    "f32 3 ragged": ("f32", 28, 4, 128, 16, [117, 117, 117], [1860, 2320, 897], "yes"),
    "f32 no hints": ("f32", 28, 4, 128, 16, [117, 117, 117], [1860, 2320, 897], "no"),
    "f32 stale hints": ("f32", 28, 4, 128, 16, [117, 30, 117], [1860, 2320, 97], "stale"),
    "f32 no workspace": ("f32", 28, 4, 128, 16, [117, 117, 117], [1860, 2320, 897], "no workspace"),
    "f16 2 ragged": ("f16", 28, 4, 128, 16, [65, 300], [6000, 31], "yes"),
    "f16 one tile, over 64 runs": ("f16", 8, 1, 128, 16, [9], [20000], "yes"),
    "f16 one step more than a tile of runs": ("f16", 32, 8, 128, 16, [130], [4000], "yes"),
    "f16 fewer steps than CUs": ("f16", 8, 2, 128, 16, [17], [1500], "yes"),
    "f16 fresh, causal tails": ("f16", 8, 2, 128, 16, [1500, 700], [0, 3], "yes"),
    "f16 d64 token pages": ("f16", 14, 2, 64, 24, [40, 200, 97], [3000, 7000, 4100], "yes"),
    "f32 d64 page 2 of 4": ("f32", 14, 2, 64, 4, [41, 77], [1000, 3100], "yes"),
    "f16 d256": ("f16", 8, 2, 256, 16, [100, 33], [2500, 900], "yes"),
    "f32 d96": ("f32", 8, 2, 96, 16, [100, 33], [2500, 900], "yes"),
    "f16 chunk behind 70 decodes": ("f16", 32, 8, 128, 16, [1] * 70 + [129], [200] * 70 + [3000], "yes"),
    "f16 chunk before 70 decodes": ("f16", 32, 8, 128, 16, [129] + [1] * 70, [3000] + [200] * 70, "no"),
}


@pytest.mark.parametrize("name", list(CASES))
def test_balanced_prefill_matches_oracle(name):
    dtype, hq, hkv, d, page, q, cached, hints = CASES[name]
    q = np.array(q, np.int32)
    seq = (np.array(cached, np.int32) + q).astype(np.int32)
    rng = np.random.default_rng(len(name))
    pages = int(sum(-(-int(L) // page) for L in seq)) + 3
    w = W.Workload(name, dtype, hq, hkv, d, page, pages, 0.3, seq, q, W._assign_pages(rng, seq, page, pages), 5)
    vals = W.host_values(w)
    t = W.device_tensors(w, vals)
    kw = {}
    if hints == "yes":
        kw = dict(seq_lens_host=w.seq_lens, cu_q_lens_host=w.cu_q_lens)
    elif hints == "stale":  # the same bounds, in another order
        kw = dict(seq_lens_host=w.seq_lens[::-1].copy(),
                  cu_q_lens_host=np.concatenate([[0], np.cumsum(q[::-1])]).astype(np.int32))
    out = torch.full((hq, w.total_q, d), float("nan"), dtype=t["q"].dtype, device="cuda")
    args = M.make_args(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"], t["cu_q_lens"], out,
                       max_q_len=w.max_q_len, max_seq_len=w.max_seq_len, sum_seq_lens=int(w.seq_lens.sum()), **kw)
    if hints != "no workspace":  # without one, the call runs unsplit
        need = M.workspace_size(args)
        ws = M.new_workspace(need, "cuda")
        args.workspace, args.workspace_bytes = ws.data_ptr(), need
    assert M.load_library().mvr_paged_attention(ctypes.byref(args)) == 0
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = O.paged_attention(vals[0], vals[1], vals[2], w.block_tables, w.seq_lens, w.cu_q_lens, hq, hkv, d, page,
                            dtype=O.F16 if dtype == "f16" else O.F32, num_threads=16)
    assert np.isfinite(got).all()
    err = float(np.abs(got - ref).max())
    print(f"[balanced prefill] {name}: max-abs vs oracle {err:.3e}", flush=True)
    assert err <= TOL[dtype], err
