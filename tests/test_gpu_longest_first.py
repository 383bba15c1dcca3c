"""GPU parity of ragged batches in 8-wavefront blocks, a block per (sequence, KV head), dispatched longest first.

The planner takes that layout from the host length tables (its calls need no workspace, which is checked), so the cases
are batches it takes: with ties, more than 64 sequences (several ranked groups, of unequal size), contexts shorter than
the block's 8 partitions, two new tokens per sequence, decodes of a mixed batch (sequences of the other launch ranked
last), stale tables (another order, still every row) and a cascade's suffix pass.  Where a call needs a workspace all
the same (mixed, cascade), its rows must not be the bits of the plan without the tables, which splits them elsewhere.
Batches that would take another plan fall back to this one in a workspace that was sized for other tables: any lengths,
any number of sequences.  Rows start as NaN; 2e-3 (F16) and 1e-5 (F32) against the oracle.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mvr_attn as M  # noqa: E402
import oracle as O  # noqa: E402
import workloads as W  # noqa: E402
from test_gpu_cascade import dev, shared_prefix_workload  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-5, "f16": 2e-3}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M.load_library()
    O.build()


def lens(n, lo, hi, seed=1):
    return np.random.default_rng(seed).integers(lo, hi, size=n, endpoint=True)


# dtype, query heads, KV heads, head_dim, new tokens per sequence, total tokens, stale tables, prefill request
CASES = {
    "f16 40": ("f16", 32, 8, 128, 1, lens(40, 500, 1400), False, 0),
    "f16 ties": ("f16", 32, 8, 128, 1, [1000, 1001, 1001, 1002] * 16, False, 0),
    "f16 67, two groups": ("f16", 16, 8, 128, 1, lens(67, 300, 1500), False, 0),
    "f16 130, three groups": ("f16", 8, 4, 128, 1, lens(130, 500, 1300), False, 0),
    "f16 short among long": ("f16", 32, 8, 128, 1, [1, 2, 16, 17, 100, 128] + [1100] * 58, False, 0),
    "f16 two tokens": ("f16", 32, 8, 128, 2, lens(36, 600, 1400), False, 0),
    "f16 stale tables": ("f16", 32, 8, 128, 1, lens(40, 500, 1400), True, 0),
    "f16 mixed": ("f16", 32, 8, 128, 1, lens(40, 500, 1400), False, 130),
    "f32 40": ("f32", 24, 8, 128, 1, lens(40, 500, 1400), False, 0),
    "f32 d64": ("f32", 32, 8, 64, 1, lens(48, 500, 1400), False, 0),
}


def attend(w, args_kw, need_workspace, workspace_bytes=None):
    host = W.host_values(w)
    t = W.device_tensors(w, host)
    out = torch.full((w.num_q_heads, w.total_q, w.head_dim), float("nan"), dtype=t["q"].dtype, device="cuda")
    args = M.make_args(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"], t["cu_q_lens"], out,
                       max_q_len=w.max_q_len, max_seq_len=w.max_seq_len, sum_seq_lens=int(w.seq_lens.sum()), **args_kw)
    need = M.workspace_size(args)
    if not need_workspace:
        assert need == 0  # one launch, merged in LDS
    if workspace_bytes is not None:
        assert need > workspace_bytes
        need = workspace_bytes
    ws = M.new_workspace(max(need, 256), "cuda")
    args.workspace, args.workspace_bytes = ws.data_ptr(), need
    assert M.load_library().mvr_paged_attention(ctypes.byref(args)) == 0
    torch.cuda.synchronize()
    return host, out.float().cpu().numpy()


def check(w, host, got, name):
    ref = O.paged_attention(host[0], host[1], host[2], w.block_tables, w.seq_lens, w.cu_q_lens, w.num_q_heads,
                            w.num_kv_heads, w.head_dim, w.page_size, dtype=O.F16 if w.dtype == "f16" else O.F32,
                            num_threads=16)
    assert np.isfinite(got).all()
    err = float(np.abs(got - ref).max())
    print(f"[longest first] {name}: max-abs vs oracle {err:.3e}", flush=True)
    assert err <= TOL[w.dtype], err


@pytest.mark.parametrize("name", list(CASES))
def test_longest_first_matches_oracle(name):
    dtype, hq, hkv, d, new, seq, stale, chunk = CASES[name]
    seq = np.array(seq, np.int32)
    q = np.full(len(seq), new, np.int32)
    if chunk:
        seq, q = np.insert(seq, 7, chunk + 300).astype(np.int32), np.insert(q, 7, chunk).astype(np.int32)
    pages = int(sum(-(-int(L) // 16) for L in seq)) + 3
    w = W.Workload(name, dtype, hq, hkv, d, 16, pages, 0.3, seq, q,
                   W._assign_pages(np.random.default_rng(2), seq, 16, pages), 5)
    host_seq = w.seq_lens[::-1].copy() if stale else w.seq_lens
    host, got = attend(w, dict(seq_lens_host=host_seq, cu_q_lens_host=w.cu_q_lens), need_workspace=bool(chunk))
    check(w, host, got, name)
    if chunk:
        _, other = attend(w, dict(cu_q_lens_host=w.cu_q_lens), need_workspace=True)
        assert not np.array_equal(got[:, :7], other[:, :7])


# dtype, total tokens, tables in the call
FALLBACK = {
    "f16 two long": ("f16", [4096, 3104] + list(lens(50, 300, 900)), "both"),
    "f16 two long, no tables": ("f16", [4096, 3104] + list(lens(50, 300, 900)), "none"),
    "f32 two long": ("f32", [4096, 3104] + list(lens(50, 300, 900)), "both"),
    "f16 equal lengths": ("f16", [1600] * 48, "both"),
    "f16 few": ("f16", [1, 700, 5000], "both"),
    "f16 one": ("f16", [5000], "none"),
    "f16 short": ("f16", lens(200, 1, 90), "both"),
}


@pytest.mark.parametrize("name", list(FALLBACK))
def test_workspace_sized_for_other_tables(name):
    dtype, seq, tables = FALLBACK[name]
    seq = np.array(seq, np.int32)
    pages = int(sum(-(-int(L) // 16) for L in seq)) + 3
    w = W.Workload(name, dtype, 32, 8, 128, 16, pages, 0.3, seq, np.ones(len(seq), np.int32),
                   W._assign_pages(np.random.default_rng(2), seq, 16, pages), 5)
    kw = dict(seq_lens_host=w.seq_lens, cu_q_lens_host=w.cu_q_lens) if tables == "both" else {}
    host, got = attend(w, kw, need_workspace=True, workspace_bytes=0)
    check(w, host, got, name)


def test_cascade_suffix_longest_first():
    members, prefix = 40, 2048
    cached = prefix + lens(members, 500, 1400)
    w = shared_prefix_workload("f16", 128, 16, [1] * members, cached, [(0, members, prefix)], hq=16, hkv=8)
    host = W.host_values(w)
    t = W.device_tensors(w, host)
    tables = [dev(x) for x in (np.array([0, members], np.int32), np.array([prefix], np.int32),
                               w.block_tables[:1].copy(), np.full(members, prefix, np.int32))]
    groups = M.make_cascade_groups(*tables, max_group_q_len=members, max_prefix_len=prefix,
                                   sum_prefix_lens=prefix * members)
    outs = []
    for kw in (dict(seq_lens_host=w.seq_lens, cu_q_lens_host=w.cu_q_lens), {}):
        out = torch.full((w.num_q_heads, w.total_q, w.head_dim), float("nan"), dtype=t["q"].dtype, device="cuda")
        args = M.make_args(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"], t["cu_q_lens"], out,
                           max_q_len=1, max_seq_len=w.max_seq_len, sum_seq_lens=int(w.seq_lens.sum()), **kw)
        lib = M.load_library()
        need = lib.mvr_paged_attention_cascade_workspace_size(ctypes.byref(args), ctypes.byref(groups))
        ws = M.new_workspace(need, "cuda")
        args.workspace, args.workspace_bytes = ws.data_ptr(), need
        assert lib.mvr_paged_attention_cascade(ctypes.byref(args), ctypes.byref(groups)) == 0
        torch.cuda.synchronize()
        outs.append(out.float().cpu().numpy())
    check(w, host, outs[0], "cascade suffix")
    assert not np.array_equal(*outs)  # the plan without the tables is another one
