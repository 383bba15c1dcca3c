"""A launch planned for shorter contexts than its device tables hold: the context splits into as many, longer
partitions, and every row is still computed (hints cost speed, never rows).  The cascade's suffix pass plans from
sum_prefix_lens = num_seqs x max_prefix_len that every sequence starts at the longest prefix; here one sequence of the
batch has no prefix at all.  F16 2e-3, F32 1e-5 against the oracle; ragged (slot == partition), dense (40 sequences)
and uniform suffixes (block merge)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mvr_attn as M  # noqa: E402
import oracle as O  # noqa: E402
import workloads as W  # noqa: E402
from test_gpu_cascade import dev, shared_prefix_workload  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M.load_library()
    O.build()


@pytest.mark.parametrize("dtype,d", [("f16", 128), ("f32", 64), ("f16", 96)])
@pytest.mark.parametrize("members,lo,hi", [(6, 600, 2900), (40, 600, 2900), (6, 2999, 2999)])
def test_sequence_without_the_planned_prefix(dtype, d, members, lo, hi):
    prefix = 512
    cached = list(np.random.default_rng(members).integers(lo, hi, size=members, endpoint=True)) + [2999]
    w = shared_prefix_workload(dtype, d, 16, [1] * (members + 1), cached, [(0, members, prefix)])
    host = W.host_values(w)
    t = W.device_tensors(w, host)
    tables = [dev(x) for x in (np.array([0, members], np.int32), np.array([prefix], np.int32),
                               w.block_tables[:1].copy(), np.array([prefix] * members + [0], np.int32))]
    groups = M.make_cascade_groups(*tables, max_group_q_len=members, max_prefix_len=prefix,
                                   sum_prefix_lens=prefix * (members + 1))
    out = M.paged_attention_cascade(t["q"], t["key_pool"], t["value_pool"], t["block_tables"], t["seq_lens"],
                                    t["cu_q_lens"], groups, max_q_len=1, max_seq_len=w.max_seq_len,
                                    sum_seq_lens=int(w.seq_lens.sum()))
    torch.cuda.synchronize()
    q, k, v = host
    ref = O.paged_attention(q, k, v, w.block_tables, w.seq_lens, w.cu_q_lens, w.num_q_heads, w.num_kv_heads, d, 16,
                            dtype=O.F16 if dtype == "f16" else O.F32, num_threads=16)
    err = float(np.abs(out.float().cpu().numpy() - ref).max())
    print(f"[planned context] {dtype} D={d} {members} members: max-abs vs oracle {err:.3e}", flush=True)
    assert err <= (2e-3 if dtype == "f16" else 1e-5), err

