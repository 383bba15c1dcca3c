"""GPU parity of the prefill kernel's main grid with every row tile's keys in the same number of parts (sequences of one
length, few unequal ones, or no host tables): parts found from the block index, merged from fp32 partials.

Cases at the places where parts can go wrong: one key tile more or less than a whole number of parts, parts of less
than a step, up to 32 parts (several rounds of the merge's 8, and of the 4 that wide F32 rows keep), fresh prompts whose
early rows see fewer key tiles than there are parts, 12 (sequence, KV head) pairs on 8 XCDs, chunks among decodes
(sequences of the other launch in the grid's range), device tables that differ from the host's, a workspace for fewer
parts or none, one-group blocks (head_dim > 128), token pages.  Rows start as NaN; 1e-5 (F32) / 2e-3 (F16) against the
oracle.
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


# dtype, query heads, KV heads, head_dim, page size, new tokens, cached tokens, hints, share of the workspace
CASES = {
    "f16 one chunk": ("f16", 28, 4, 128, 16, [100], [4289], "yes", 1),
    "f16 no tables": ("f16", 28, 4, 128, 16, [100], [4289], "no", 1),
    "f16 tile boundary": ("f16", 8, 2, 128, 16, [64], [64 * 31], "yes", 1),
    "f16 one past it": ("f16", 8, 2, 128, 16, [64], [64 * 31 + 1], "yes", 1),
    "f16 half steps": ("f16", 8, 2, 128, 16, [20], [900], "yes", 1),
    "f16 one tile, 32 parts": ("f16", 8, 1, 128, 16, [9], [20000], "yes", 1),
    "f16 12 pairs": ("f16", 28, 4, 128, 16, [50] * 3, [3000] * 3, "yes", 1),
    "f16 fresh": ("f16", 2, 1, 128, 16, [2000], [0], "yes", 1),
    "f16 near-fresh pair": ("f16", 2, 1, 128, 16, [1700] * 2, [3] * 2, "yes", 1),
    "f16 other device tables": ("f16", 32, 8, 128, 16, [100, 37, 64], [40, 2100, 900], "equal", 1),
    "f16 half the workspace": ("f16", 28, 4, 128, 16, [100], [4289], "yes", 0.5),
    "f16 no workspace": ("f16", 28, 4, 128, 16, [100], [4289], "yes", 0),
    "f16 chunks among decodes": ("f16", 32, 8, 128, 16, [1, 130, 1, 1, 130, 1], [90, 2000, 700, 5, 2000, 300], "yes", 1),
    "f16 chunk among decodes, no tables": ("f16", 32, 8, 128, 16, [1, 130, 1, 1], [90, 2000, 700, 5], "no", 1),
    "f16 130 on 4000": ("f16", 32, 8, 128, 16, [130], [4000], "yes", 1),
    "f16 17 on 1500": ("f16", 8, 2, 128, 16, [17], [1500], "yes", 1),
    "f16 chunk behind 70 decodes": ("f16", 32, 8, 128, 16, [1] * 70 + [129], [200] * 70 + [3000], "yes", 1),
    "f16 chunk before 70 decodes, no tables": ("f16", 32, 8, 128, 16, [129] + [1] * 70, [3000] + [200] * 70, "no", 1),
    "f16 d64 unequal, token pages": ("f16", 14, 2, 64, 24, [40, 200, 97], [3000, 7000, 4100], "yes", 1),
    "f32 d64 unequal, 4-token pages": ("f32", 14, 2, 64, 4, [41, 77], [1000, 3100], "yes", 1),
    "f16 d256 unequal": ("f16", 8, 2, 256, 16, [100, 33], [2500, 900], "yes", 1),
    "f32 d96 unequal": ("f32", 8, 2, 96, 16, [100, 33], [2500, 900], "yes", 1),
    "f32 unequal, no tables": ("f32", 32, 8, 128, 16, [117] * 3, [1860, 2320, 897], "no", 1),
    "f16 d64": ("f16", 14, 2, 64, 16, [256], [2048], "yes", 1),
    "f16 d64 token pages": ("f16", 14, 2, 64, 24, [97] * 2, [3000] * 2, "yes", 1),
    "f16 d128 4-token pages": ("f16", 8, 2, 128, 4, [70], [3001], "yes", 1),
    "f16 d96": ("f16", 8, 2, 96, 16, [100], [3000], "yes", 1),
    "f16 d256": ("f16", 8, 2, 256, 16, [100], [3000], "yes", 1),
    "f32 one chunk": ("f32", 28, 4, 128, 16, [100], [4289], "yes", 1),
    "f32 several rounds": ("f32", 32, 8, 128, 16, [99] * 3, [700] * 3, "yes", 1),
    "f32 d64": ("f32", 32, 8, 64, 16, [100], [3000], "yes", 1),
    "f32 d64 2-token pages": ("f32", 14, 2, 64, 4, [77], [1001], "yes", 1),
    "f32 d160": ("f32", 8, 2, 160, 16, [40], [1700], "yes", 1),
    "f32 d192": ("f32", 8, 2, 192, 16, [40], [1100], "yes", 1),
    "f32 d224, 32 parts": ("f32", 8, 2, 224, 16, [64], [8000], "no", 1),
    "f32 d224, few parts": ("f32", 8, 2, 224, 16, [33], [190], "yes", 1),
    "f32 d256": ("f32", 8, 2, 256, 16, [40], [2100], "yes", 1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prefill_in_equal_parts_matches_oracle(name):
    dtype, hq, hkv, d, page, q, cached, hints, share = CASES[name]
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
    elif hints == "equal":  # every sequence at the call's bounds
        kw = dict(seq_lens_host=np.full(len(q), w.max_seq_len, np.int32),
                  cu_q_lens_host=(np.arange(len(q) + 1) * w.max_q_len).astype(np.int32))
    out = torch.full((hq, w.total_q, d), float("nan"), dtype=t["q"].dtype, device="cuda")
    args = M.make_args(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"], t["cu_q_lens"], out,
                       max_q_len=w.max_q_len, max_seq_len=w.max_seq_len, **kw)
    need = M.workspace_size(args)
    assert need > 0  # partials: the call is split
    need = int(need * share)
    ws = M.new_workspace(max(need, 256), "cuda")
    ws.fill_(255)  # NaN in every part that this call does not write: none may reach the rows
    args.workspace, args.workspace_bytes = ws.data_ptr(), need
    assert M.load_library().mvr_paged_attention(ctypes.byref(args)) == 0, M.load_library().mvr_last_error()
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = O.paged_attention(vals[0], vals[1], vals[2], w.block_tables, w.seq_lens, w.cu_q_lens, hq, hkv, d, page,
                            dtype=O.F16 if dtype == "f16" else O.F32, num_threads=16)
    assert np.isfinite(got).all()
    err = float(np.abs(got - ref).max())
    print(f"[prefill parts] {name}: max-abs vs oracle {err:.3e}", flush=True)
    assert err <= TOL[dtype], err
