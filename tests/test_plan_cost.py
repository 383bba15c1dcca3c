"""What planning a call costs the host, paid for each layer: a pass or two over the batch's length tables, not a pass for
each part count that the planner tries.  Measured as the growth from 500 to 4,000 sequences, on the sizing call, which
runs the same planner."""
import ctypes
import os
import time

import numpy as np
import pytest

import mvr_attn as M

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-vllm-rs_amd", "libmvr_attn.so")


def call(n, chunk):
    a = M.PagedAttentionArgs()
    q = np.ones(n, np.int32)
    if chunk:
        q[-1] = chunk
    seq = (np.full(n, 2000) + q).astype(np.int32)
    cu = np.concatenate([[0], np.cumsum(q)]).astype(np.int32)
    a.dtype, a.num_seqs, a.num_q_heads, a.num_kv_heads, a.head_dim = M.DTYPE_F16, n, 32, 8, 128
    a.page_size, a.num_pages, a.max_pages_per_seq = 16, 1 << 20, 256
    a.max_q_len, a.max_seq_len, a.sum_seq_lens = int(q.max()), int(seq.max()), int(seq.sum())
    a.q = a.key_pool = a.value_pool = a.block_tables = a.seq_lens = a.cu_q_lens = a.out = 1 << 32
    a.q_stride_head, a.q_stride_token, a.out_stride_head, a.out_stride_token = 1 << 20, 128, 1 << 20, 128
    a.seq_lens_host, a.cu_q_lens_host = seq.ctypes.data, cu.ctypes.data
    a._keep = seq, cu
    return a


def seconds(n, chunk):
    lib, a = M.load_library(), call(n, chunk)
    ref = ctypes.byref(a)
    best = 1.0
    for _ in range(30):
        t = time.perf_counter()
        for _ in range(20):
            lib.mvr_paged_attention_workspace_size(ref)
        best = min(best, (time.perf_counter() - t) / 20)
    return best


def test_planning_a_mixed_call_reads_the_tables_a_few_times():
    if not os.path.exists(LIB):
        pytest.skip("build the library first (python -c 'import __graft_entry__ as g; g.build()')")
    per_seq = (seconds(4000, 256) - seconds(500, 256)) / 3500 * 1e9
    print(f"[plan cost] {per_seq:.2f} ns per sequence of a mixed call")
    # One pass over both tables with its checks takes about 4 ns a sequence, sixty took 38.
    assert per_seq < 15
