"""GPU parity of the prefill kernel's balanced grid: each row tile's keys in parts of about one length, a block per
part, found from the device length tables, and a merge of the tiles that have several.

The planner takes it for sequences of unequal lengths, and for (sequence, KV head) pairs that the 8 XCDs share
unevenly, where a block per 128-row tile leaves CUs idle or waits for the longest.  Cases at the places where parts can go wrong: one and many parts per tile (over several rounds of the merge's
8, and of the 4 that F32 keeps, up to 32), causal limits that leave a tile fewer key tiles than parts, more than 64
sequences (the device scan's second round) with decodes among them, device tables that give more parts, or more tiles,
than the host's did (the call then runs unsplit, its blocks striding over whole tiles), no workspace, token pages,
one-group blocks (head_dim > 128).  Each case names the grid it takes, which the planner's CPU test checks.  Every
output row must be written and meet 1e-5 (F32) / 2e-3 (F16) against the oracle.
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


# dtype, query heads, KV heads, head_dim, page size, new tokens, cached tokens, host tables (the device's; none; no
# workspace; or other ones), grid: balanced, unsplit (more parts than planned), strided (several tiles per block)
CASES = {
    "f32 3 ragged": ("f32", 28, 4, 128, 16, [117, 117, 117], [1860, 2320, 897], "tables", "balanced"),
    "f32 no workspace": ("f32", 28, 4, 128, 16, [117, 117, 117], [1860, 2320, 897], "no workspace", "unsplit"),
    "f32 one length, 12 pairs": ("f32", 28, 4, 128, 16, [99] * 3, [700] * 3, "tables", "balanced"),
    "f32 other order": ("f32", 28, 4, 128, 16, [117, 30, 117], [1860, 2320, 97], "reversed", "balanced"),
    "f32 more parts": ("f32", 28, 4, 128, 16, [60, 60, 60], [3440, 3440, 2000], "one long", "more parts"),
    "f16 more parts": ("f16", 28, 4, 128, 16, [60, 60, 60], [3440, 3440, 2000], "one long", "more parts"),
    "f16 more tiles": ("f16", 32, 8, 128, 16, [300] * 8, [500, 3000, 77, 900, 2000, 1234, 64, 0], "one long of 8", "strided"),
    "f32 d64 more tiles": ("f32", 32, 8, 64, 16, [300] * 8, [500, 3000, 77, 900, 20, 1234, 64, 0], "one long of 8", "strided"),
    "f16 d256 more tiles": ("f16", 32, 8, 256, 16, [300] * 8, [500, 3000, 77, 900, 200, 1234, 64, 0], "one long of 8", "strided"),
    "f16 2 ragged": ("f16", 28, 4, 128, 16, [65, 300], [6000, 31], "tables", "balanced"),
    "f16 past 8 parts": ("f16", 8, 1, 128, 16, [59, 85], [3552, 50], "tables", "balanced"),
    "f16 causal": ("f16", 8, 1, 128, 16, [538, 83], [17, 5602], "tables", "balanced"),
    "f16 fresh, causal tails": ("f16", 8, 2, 128, 16, [1500, 700], [0, 3], "tables", "balanced"),
    "f16 d64 token pages, past 8 parts": ("f16", 14, 2, 64, 24, [78, 18], [68, 4738], "tables", "balanced"),
    "f32 d64 4-token pages, past 8 parts": ("f32", 14, 2, 64, 4, [12, 37], [2102, 117], "tables", "balanced"),
    "f32 d64 causal": ("f32", 14, 2, 64, 16, [260, 118], [11, 1227], "tables", "balanced"),
    "f16 d256, past 8 parts": ("f16", 8, 2, 256, 16, [90, 17], [144, 2113], "tables", "balanced"),
    "f32 d96, past 8 parts": ("f32", 8, 2, 96, 16, [31, 101], [2335, 253], "tables", "balanced"),
    "f32 d160, past 4 parts": ("f32", 8, 2, 160, 16, [73, 27], [65, 1181], "tables", "balanced"),
    "f32 d192, past 4 parts": ("f32", 8, 2, 192, 16, [12, 134], [891, 74], "tables", "balanced"),
    "f32 d224, past 4 parts": ("f32", 8, 2, 224, 16, [29, 43], [1564, 193], "tables", "balanced"),
    "f32 d256, past 4 parts": ("f32", 8, 2, 256, 16, [16, 49], [1055, 108], "tables", "balanced"),
    "f16 two chunks behind 70 decodes": ("f16", 32, 8, 128, 16, [1] * 70 + [129, 70], [200] * 70 + [3000, 600], "tables",
                                         "balanced"),
    "f16 two chunks before 70 decodes": ("f16", 32, 8, 128, 16, [129, 70] + [1] * 70, [3000, 600] + [200] * 70, "tables",
                                         "balanced"),
}


def host_tables(kind):
    """(new tokens, total tokens) of host tables that are not the device's, within the call's bounds."""
    q, seq = {
        "reversed": ([117, 30, 117], [214, 2350, 1977]),
        "one long": ([57, 36, 36], [132, 3500, 132]),
        "one long of 8": ([40] + [10] * 7, [3300] + [90] * 7),
    }[kind]
    return np.array(q, np.int32), np.array(seq, np.int32)


@pytest.mark.parametrize("name", list(CASES))
def test_balanced_prefill_matches_oracle(name):
    dtype, hq, hkv, d, page, q, cached, host, grid = CASES[name]
    q = np.array(q, np.int32)
    seq = (np.array(cached, np.int32) + q).astype(np.int32)
    rng = np.random.default_rng(len(name))
    pages = int(sum(-(-int(L) // page) for L in seq)) + 3
    w = W.Workload(name, dtype, hq, hkv, d, page, pages, 0.3, seq, q, W._assign_pages(rng, seq, page, pages), 5)
    vals = W.host_values(w)
    t = W.device_tensors(w, vals)
    kw = {}
    if host in ("tables", "no workspace"):
        kw = dict(seq_lens_host=w.seq_lens, cu_q_lens_host=w.cu_q_lens)
    elif host != "none":
        host_q, host_seq = host_tables(host)
        kw = dict(seq_lens_host=host_seq, cu_q_lens_host=np.concatenate([[0], np.cumsum(host_q)]).astype(np.int32))
    out = torch.full((hq, w.total_q, d), float("nan"), dtype=t["q"].dtype, device="cuda")
    args = M.make_args(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"], t["cu_q_lens"], out,
                       max_q_len=w.max_q_len, max_seq_len=w.max_seq_len, sum_seq_lens=int(w.seq_lens.sum()), **kw)
    if host != "no workspace":
        need = M.workspace_size(args)
        assert need > 0  # partials: the call is split
        ws = M.new_workspace(need, "cuda")
        ws.fill_(255)  # NaN in every part that this call does not write
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
