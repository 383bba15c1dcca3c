"""A workspace sized once with hints serves every later call of the same scalar fields, whatever the host tables hold
by then: lengths shift between steps, and a plan that suits the new ones may want more than the old ones did.

On the CPU the calls stop at the launch (MVR_E_HIP: there is no device), after the workspace check, and the dummy
addresses are never read; where there is a GPU these tests do not run (test_gpu_longest_first.py makes such calls on
real tensors)."""
import ctypes

import numpy as np
import pytest

import mvr_attn as M

FAKE = 1 << 32


@pytest.fixture(autouse=True)
def _no_device():
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("the calls below carry dummy addresses")


def args(seq, q=None, tables=True, dtype=M.DTYPE_F16, total=None, hq=32, hkv=8, d=128, page=16, max_seq_len=8192,
         max_q_len=None):
    q = np.ones(len(seq), np.int32) if q is None else np.asarray(q, np.int32)
    a = M.PagedAttentionArgs()
    a.dtype, a.num_seqs, a.num_q_heads, a.num_kv_heads, a.head_dim = dtype, len(seq), hq, hkv, d
    a.page_size, a.num_pages, a.max_pages_per_seq = page, 1 << 20, -(-max_seq_len // page)
    a.max_q_len, a.max_seq_len = int(max_q_len or q.max()), max_seq_len
    a.q = a.key_pool = a.value_pool = a.block_tables = a.seq_lens = a.cu_q_lens = a.out = FAKE
    a.q_stride_head, a.q_stride_token, a.out_stride_head, a.out_stride_token = 8192 * d, d, 8192 * d, d
    a.sum_seq_lens = int(np.sum(seq)) if total is None else total
    a._keep = (np.ascontiguousarray(seq, np.int32), np.concatenate([[0], np.cumsum(q)]).astype(np.int32))
    if tables:
        a.seq_lens_host, a.cu_q_lens_host = (x.ctypes.data for x in a._keep)
    return a


def call(a, workspace_bytes):
    lib = M.load_library()
    a.workspace, a.workspace_bytes = (FAKE if workspace_bytes else 0), workspace_bytes
    rc = lib.mvr_paged_attention(ctypes.byref(a))
    return rc, lib.mvr_last_error().decode()


EVEN = [1500] * 60 + [1400, 1600] * 2
TWO_LONG = [8192, 7208] + [1300] * 62


@pytest.mark.parametrize("dtype", [M.DTYPE_F16, M.DTYPE_F32])
@pytest.mark.parametrize("tables", [True, False])
def test_decode_workspace_sized_for_other_tables(dtype, tables):
    assert sum(EVEN) == sum(TWO_LONG)
    even, later = args(EVEN, dtype=dtype), args(TWO_LONG, dtype=dtype, tables=tables)
    assert M.workspace_size(even) < M.workspace_size(later)  # else this test shows nothing
    rc, err = call(later, M.workspace_size(even))
    assert rc == M.MVR_E_HIP, err
    # Sized without the tables, it holds the plan of any of them.
    assert M.workspace_size(args(EVEN, dtype=dtype, tables=False)) == M.workspace_size(args(TWO_LONG, dtype=dtype))


def test_equal_lengths_after_ragged_ones():
    ragged, equal = args([1500] * 46 + [1400, 1600], max_seq_len=1600), args([1600] * 48, max_seq_len=1600)
    assert M.workspace_size(ragged) < M.workspace_size(equal)
    rc, err = call(equal, M.workspace_size(ragged))
    assert rc == M.MVR_E_HIP, err


def test_mixed_workspace_sized_for_other_tables():
    q = [1] * 64 + [256]
    even, later = args(EVEN + [2304], q), args(TWO_LONG + [2304], q)
    assert M.workspace_size(even) < M.workspace_size(later)
    rc, err = call(later, M.workspace_size(even))
    assert rc == M.MVR_E_HIP, err


def test_cascade_workspace_does_not_depend_on_the_tables():
    lib = M.load_library()
    g = M.CascadeGroups()
    g.num_groups, g.max_group_q_len, g.max_prefix_len, g.sum_prefix_lens = 1, 64, 512, 512 * 64
    g.group_cu_q_lens = g.group_prefix_lens = g.group_block_tables = g.seq_prefix_lens = FAKE
    even, later = (args(512 + np.array(x), max_seq_len=8704) for x in (EVEN, TWO_LONG))
    need = [lib.mvr_paged_attention_cascade_workspace_size(ctypes.byref(a), ctypes.byref(g)) for a in (even, later)]
    assert need[0] == need[1]
    later.workspace, later.workspace_bytes = FAKE, need[0]
    rc = lib.mvr_paged_attention_cascade(ctypes.byref(later), ctypes.byref(g))
    assert rc == M.MVR_E_HIP, lib.mvr_last_error().decode()


@pytest.mark.parametrize("seq,kw", [([1600] * 48, dict(total=0, tables=False, max_seq_len=1600)),
                                    (TWO_LONG, dict(d=64)), (TWO_LONG, dict(page=8))])
def test_plans_that_need_partials_still_refuse_less(seq, kw):
    a = args(seq, **kw)
    need = M.workspace_size(a)
    rc, err = call(a, need - 1)
    assert need > 0 and rc == M.MVR_E_WORKSPACE and "smaller than" in err
