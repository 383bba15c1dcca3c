"""The prefill plans that the GPU parity tests of split grids mean to run, read from the planner on the CPU: their cases
state the grid they take, so a case cannot drift to another plan unnoticed.  The planner's source is compiled into a
program that prints each case's plan for 256 CUs; nothing is launched."""
import os
import shutil
import subprocess

import numpy as np
import pytest

pytest.importorskip("torch")

import test_gpu_prefill_balanced as B  # noqa: E402
import test_gpu_prefill_parts as P  # noqa: E402

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mini-vllm-rs_amd")
HIPCC = "/opt/rocm/bin/hipcc"
OBJS = [os.path.join(PKG, "_build", o) for o in ("paged_attention.o", "paged_prefill.o", "kv_gather.o", "kv_append.o")]

PROGRAM = r"""
#include "mvr_attn_api.cpp"
// Lines of: dtype hq hkv d page max_q max_seq tables workspace n, then n q_lens and n seq_lens.
int main() {
  int dtype, hq, hkv, d, page, max_q, max_seq, tables, n;
  long long ws;
  while (scanf("%d %d %d %d %d %d %d %d %lld %d", &dtype, &hq, &hkv, &d, &page, &max_q, &max_seq, &tables, &ws, &n) == 10) {
    std::vector<int32_t> cu(n + 1), seq(n);
    for (int i = 0; i < n; i++) { scanf("%d", &cu[i + 1]); cu[i + 1] += cu[i]; }
    for (int i = 0; i < n; i++) scanf("%d", &seq[i]);
    mvr_paged_attention_args a{};
    a.dtype = dtype; a.num_seqs = n; a.num_q_heads = hq; a.num_kv_heads = hkv; a.head_dim = d; a.page_size = page;
    a.max_pages_per_seq = 1 << 20; a.num_pages = 1 << 20; a.max_q_len = max_q; a.max_seq_len = max_seq;
    if (tables) { a.seq_lens_host = seq.data(); a.cu_q_lens_host = cu.data(); }
    else a.total_q = cu[n];
    const CallPlan c = make_call_plan(&a, ws < 0 ? SIZE_MAX : (size_t)ws);
    const mvr::PagedAttentionPlan& p = c.plan[c.n - 1];
    printf("%d %d %d %d %d %d %d\n", c.n, (int)p.prefill, p.kv_splits, p.balanced_blocks, p.balanced_tiles, p.part_steps,
           prefill_step_keys(&a));
  }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if not os.path.exists(HIPCC) or not all(os.path.exists(o) for o in OBJS):
        pytest.skip("needs hipcc and the built library (python -c 'import __graft_entry__ as g; g.build()')")
    if shutil.which("rocminfo") and os.path.exists("/dev/kfd"):
        pytest.skip("plans depend on the CUs of a present device")
    tmp = tmp_path_factory.mktemp("plans")
    src, exe = tmp / "plans.cpp", tmp / "plans"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-w", "-fPIC",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"), "-c", str(src), "-o",
                    str(tmp / "plans.o")], check=True, capture_output=True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", str(tmp / "plans.o"), *OBJS, "-o", str(exe), "-L/opt/rocm/lib",
                    "-lrocprofiler-sdk-roctx", "-Wl,-rpath,/opt/rocm/lib"], check=True, capture_output=True)

    def run(dtype, hq, hkv, d, page, max_q, max_seq, tables, q, seq, workspace=-1):
        line = [dtype == "f16", hq, hkv, d, page, max_q, max_seq, tables, workspace, len(q), *q, *seq]
        r = subprocess.run([str(exe)], input=" ".join(str(int(x)) for x in line) + "\n", capture_output=True, text=True,
                           check=True)
        return dict(zip(("launches", "prefill", "kv_splits", "blocks", "tiles", "part_steps", "step_keys"),
                        map(int, r.stdout.split())))

    return run


@pytest.mark.parametrize("name", list(P.CASES))
def test_equal_parts(plan, name):
    dtype, hq, hkv, d, page, q, cached, hints, share = P.CASES[name]
    seq = np.array(cached) + q
    tables = {"yes": (q, seq), "no": (q, seq), "equal": ([max(q)] * len(q), [max(seq)] * len(q))}[hints]
    p = plan(dtype, hq, hkv, d, page, max(q), max(seq), hints != "no", *tables, workspace=0 if share == 0 else -1)
    assert p["prefill"] and p["blocks"] == 0
    assert (p["kv_splits"] > 1) == (share > 0), p
    if "32 parts" in name:
        assert p["kv_splits"] == 32, p


@pytest.mark.parametrize("name", list(B.CASES))
def test_balanced(plan, name):
    dtype, hq, hkv, d, page, q, cached, host, grid = B.CASES[name]
    q, seq = np.array(q), np.array(cached) + q
    host_q, host_seq = (q, seq) if host in ("tables", "no workspace") else B.host_tables(host)
    p = plan(dtype, hq, hkv, d, page, max(q), max(seq), host != "none", *((q, seq) if host == "none" else (host_q, host_seq)),
             workspace=0 if host == "no workspace" else -1)
    assert p["prefill"]
    if grid == "unsplit":
        assert p["blocks"] == 0 and p["kv_splits"] == 1, p
        return
    assert p["blocks"] > 0 and p["kv_splits"] == 1, p
    # What the device makes of its tables: parts per tile from each sequence's steps.
    rows = hq // hkv * q
    rows[q <= 32 // (hq // hkv)] = 0 if p["launches"] == 2 else rows[q <= 32 // (hq // hkv)]
    tiles = hkv * -(-rows // 128)
    steps = -(-seq // p["step_keys"])
    parts = np.minimum(-(-steps // p["part_steps"]), 32)
    fits = (tiles * parts).sum() <= p["blocks"] and tiles.sum() <= p["tiles"]
    assert fits == (grid == "balanced"), (p, tiles, parts)
    if grid == "strided":  # the fallback's blocks take several tiles each
        assert tiles.sum() >= 2 * p["blocks"], (p, tiles)
    if "causal" in name:  # the first row tile sees fewer steps than there are parts
        assert (parts[0] > -(-128 // p["step_keys"])) and parts[0] > 1, (p, parts)
    if "past 4" in name:
        assert parts.max() > 4 and parts.max() % 4, (p, parts)
    if "past 8" in name:
        assert parts.max() > 8 and parts.max() % 8, (p, parts)


def test_many_lengths(plan):
    """As many different lengths as a splittable call can have (4 row tiles per CU) are all planned."""
    n = 500
    seq = 300 + 130 * (np.arange(n) % 40) + 4000 * (np.arange(n) % 37 == 0)
    p = plan("f32", 4, 1, 128, 16, 30, int(seq.max()), True, [30] * n, seq)
    assert p["blocks"] > n, p


# Row tiles near or past the CUs: dtype, heads, KV heads, head_dim, new tokens, cached tokens, grid.
GRIDS = {
    "f32 480 tiles": ("f32", 32, 8, 64, [627] * 3, [679, 428, 878], "unsplit"),
    "f16 352 tiles": ("f16", 32, 8, 128, [700] * 2, [4888, 605], "unsplit"),
    "f16 144 tiles": ("f16", 24, 8, 128, [119] * 6, [3543, 2990, 3425, 3645, 3113, 1695], "unsplit"),
    "f16 one sequence, 56 tiles": ("f16", 28, 4, 128, [256], [2048], "parts"),
    "f32 160 tiles of one length": ("f32", 32, 8, 128, [151] * 4, [1593] * 4, "parts"),
    "f32 12 pairs of one length": ("f32", 28, 4, 128, [151] * 3, [1593] * 3, "balanced"),
}


@pytest.mark.parametrize("name", list(GRIDS))
def test_grids_of_many_tiles(plan, name):
    """More blocks than CUs run in rounds, each as long as a part: only where that is shorter is a call split."""
    dtype, hq, hkv, d, q, cached, grid = GRIDS[name]
    seq = np.array(cached) + q
    p = plan(dtype, hq, hkv, d, 16, max(q), int(seq.max()), True, q, seq)
    assert p["prefill"]
    assert ("balanced" if p["blocks"] else "parts" if p["kv_splits"] > 1 else "unsplit") == grid, p
