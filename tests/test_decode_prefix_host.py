"""The step prefix that every decode workgroup builds, run on the CPU: the device functions'
own text (seq_steps, fill_row, build_step_prefix of paged_decode.hip) is compiled for the host
with one thread per work item, and a block table that records which entries are read.

The entry points promise that block-table entries at index >= ceil(context / block_size) are
never read, so a row without steps (context 0, or an impossible length) has no readable entry:
a caller may leave such rows without memory behind them.  A read there is visible only here,
since the value is not used.
"""

import re
import shutil
import subprocess

import pytest

from kavor_amd._build import CSRC_DIR

FUNCTIONS = ["seq_steps", "fill_row", "build_step_prefix"]

SHIM = r"""
#include <algorithm>
#include <barrier>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <set>
#include <thread>
#include <vector>
using std::max;
using std::min;
typedef uint32_t u32;
#define __device__
#define __forceinline__ inline
constexpr int kDecodeHeadDim = 128, kDecodeWaves = 4, kDecodeThreads = 256, kStep = 32;
struct uint4 { u32 x, y, z, w; };
static uint4 make_uint4(u32 x, u32 y, u32 z, u32 w) { return {x, y, z, w}; }
struct Index { int x, y; };
static thread_local Index threadIdx;
static Index blockIdx{0, 0}, gridDim{1, 1};
static std::barrier<> all(kDecodeThreads);
static void __syncthreads() { all.arrive_and_wait(); }
static int scan_in[kDecodeThreads];
static int wave_incl_scan(int x) {
  scan_in[threadIdx.x] = x;
  __syncthreads();
  int sum = 0;
  for (int t = threadIdx.x & ~63; t <= threadIdx.x; ++t) sum += scan_in[t];
  __syncthreads();
  return sum;
}
static void keep(int) {}
struct Table {  // records the entries that are read
  std::set<int64_t>* seen;
  std::mutex* lock;
  int operator[](int64_t i) const {
    std::lock_guard<std::mutex> g(*lock);
    seen->insert(i);
    return 0;
  }
};
struct DecodeParams {
  const int* context_lens;
  Table block_tables;
  int64_t bt_stride;
  int num_seqs, num_q_heads, max_blocks, block_size;
  uint16_t* out;
  int64_t o_seq_stride, o_head_stride;
};
"""

MAIN = r"""
int main(int argc, char** argv) {  // stride, max_blocks, block_size, then the context lengths
  std::vector<int> ctx;
  for (int i = 4; i < argc; ++i) ctx.push_back(atoi(argv[i]));
  const int B = static_cast<int>(ctx.size());
  std::set<int64_t> seen;
  std::mutex lock;
  std::vector<uint16_t> out(B * 128, 1);
  DecodeParams p{ctx.data(), Table{&seen, &lock}, atoi(argv[1]), B, 1, atoi(argv[2]), atoi(argv[3]), out.data(), 128, 128};
  std::vector<int> s_cum(B + 1, -1);
  int s_part[kDecodeWaves];
  std::vector<std::thread> ts;
  for (int t = 0; t < kDecodeThreads; ++t)
    ts.emplace_back([&, t] {
      threadIdx = {t, 0};
      build_step_prefix(p, s_cum.data(), s_part);
    });
  for (auto& t : ts) t.join();
  for (int v : s_cum) printf("%d ", v);
  printf("\n");
  for (int64_t i : seen) printf("%lld ", static_cast<long long>(i));
  printf("\n");
  for (int b = 0; b < B; ++b) printf("%d ", out[b * 128]);
  printf("\n");
}
"""


def _function(src: str, name: str) -> str:
    """The text of one device function: from its __device__ to its closing brace."""
    start = re.search(rf"^__device__[^\n;{{}}]*\b{name}\(", src, re.M).start()
    depth, i = 0, src.index("{", start)
    while True:
        depth += {"{": 1, "}": -1}.get(src[i], 0)
        i += 1
        if depth == 0:
            return src[start:i]


@pytest.fixture(scope="module")
def prefix(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    src = (CSRC_DIR / "paged_decode.hip").read_text()
    work = tmp_path_factory.mktemp("prefix")
    (work / "p.cc").write_text(SHIM + "\n".join(_function(src, f) for f in FUNCTIONS) + MAIN)
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", "-w", "-o", str(work / "p"), str(work / "p.cc")], check=True)

    def run(ctx, stride=8, max_blocks=4, block_size=64):
        out = subprocess.run([str(work / "p"), *map(str, (stride, max_blocks, block_size, *ctx))], check=True,
                             capture_output=True, text=True, timeout=60).stdout.split("\n")
        return [[int(v) for v in line.split()] for line in out[:3]]

    return run


@pytest.mark.parametrize("ctx", [
    [0, 0, 0, 0],                                       # nothing but padding rows
    [5, 0, 64, 257, 256, -3, 33],                       # too long (257 > 4 * 64) and negative among live ones
    [(7 * b) % 200 if b % 3 else 0 for b in range(256)],
    [(11 * b) % 250 if b % 4 else 0 for b in range(300)],  # more sequences than threads
])
def test_prefix_reads_no_entry_of_a_row_without_steps(prefix, ctx):
    cum, seen, out = prefix(ctx)
    steps = [-(-c // 32) if 0 < c <= 256 else 0 for c in ctx]
    assert cum == [sum(steps[:b]) for b in range(len(ctx) + 1)]
    for i in seen:
        row, entry = divmod(i, 8)
        assert steps[row] > 0 and entry * 64 < ctx[row], f"entry {entry} of row {row} (context {ctx[row]}) was read"
    for b, c in enumerate(ctx):  # zeros for an empty row, NaN for an impossible one, else untouched
        assert out[b] == (1 if steps[b] else 0 if c <= 0 else 0x7FC0)
