"""Planning a call allocates nothing on the heap, whatever the batch (the header's promise for the launching entry
points, which plan before they launch; an allocation that fails would also throw through the C boundary).  A program
with its own operator new counts the allocations of the sizing calls, which run the same planner, with the library
loaded behind it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "mini-vllm-rs_amd", "libmvr_attn.so")

PROGRAM = r"""
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <initializer_list>
#include <new>
#include "mvr_attn.h"
static long count = 0;
void* operator new(size_t n) { count++; if (void* p = malloc(n)) return p; throw std::bad_alloc(); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main(int, char** argv) {
  void* lib = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL);
  if (!lib) { printf("%s\n", dlerror()); return 2; }
  auto size = (size_t(*)(const mvr_paged_attention_args*))dlsym(lib, "mvr_paged_attention_workspace_size");
  auto cascade = (size_t(*)(const mvr_paged_attention_args*, const mvr_cascade_groups*))dlsym(
      lib, "mvr_paged_attention_cascade_workspace_size");
  static int32_t seq[8192], cu[8193];
  void* fake = (void*)((size_t)1 << 32);
  for (int n : {1, 33, 64, 300, 5000})
    for (int dtype = 0; dtype < 2; dtype++)
      for (int chunk : {0, 200}) {
        mvr_paged_attention_args a;
        memset(&a, 0, sizeof a);
        a.dtype = dtype; a.num_seqs = n; a.num_q_heads = 32; a.num_kv_heads = 8; a.head_dim = 128;
        a.page_size = 16; a.max_pages_per_seq = 128; a.num_pages = 1 << 20; a.max_seq_len = 2048;
        a.max_q_len = chunk ? chunk : 1;
        a.q = fake; a.key_pool = fake; a.value_pool = fake; a.out = fake;
        a.block_tables = a.seq_lens = a.cu_q_lens = (const int32_t*)fake;
        a.q_stride_head = a.out_stride_head = 1 << 20; a.q_stride_token = a.out_stride_token = 128;
        for (int s = 0; s < n; s++) {
          const int q = chunk && s == n / 2 ? chunk : 1;
          seq[s] = 900 + 37 * (s % 30);
          cu[s + 1] = cu[s] + q;
          a.sum_seq_lens += seq[s];
        }
        a.seq_lens_host = seq; a.cu_q_lens_host = cu;
        mvr_cascade_groups g;
        memset(&g, 0, sizeof g);
        g.num_groups = 1; g.max_group_q_len = n; g.max_prefix_len = 512; g.sum_prefix_lens = 512L * n;
        g.group_cu_q_lens = g.group_prefix_lens = g.group_block_tables = g.seq_prefix_lens = (const int32_t*)fake;
        long sum = 0;
        for (int i = 0; i < 3; i++) {
          const long before = count;
          sum += (long)size(&a) + (long)cascade(&a, &g);
          if (i) printf("n %d dtype %d chunk %d: %ld allocations\n", n, dtype, chunk, count - before);
        }
      }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_planning_allocates_nothing(tmp_path):
    if not os.path.exists(LIB):
        pytest.skip("build the library first (python -c 'import __graft_entry__ as g; g.build()')")
    src, exe = tmp_path / "count.cpp", tmp_path / "count"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-rdynamic", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe),
                    "-ldl"], check=True)
    r = subprocess.run([str(exe), LIB], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.splitlines()
    assert len(lines) == 40
    bad = [x for x in lines if not x.endswith(": 0 allocations")]
    assert not bad, bad
