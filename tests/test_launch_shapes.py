"""Launch shapes of the persistent traversal, computed on the host: what a launch takes
of the chip fits its rays, so that launches on other streams find room beside it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "snkpt_dev.h"
using namespace snkpt;
int main(int argc, char** argv) {
    const uint32_t cus = 256;
    for (int i = 1; i + 1 < argc; i += 2) {
        const uint32_t need = (uint32_t)atoi(argv[i]), n = (uint32_t)strtoul(argv[i + 1], nullptr, 10);
        with_stack(need, [&](auto s) {
            constexpr int S = decltype(s)::value;
            const TraceGrid g = trace_grid(S, trace_waves(S), (uint32_t)cu_waves(S), cus, n);
            printf("%u %u %d %d %d %u %u\n", need, n, S, cu_waves(S), trace_waves(S), g.blocks, g.threads);
        });
    }
    return 0;
}
"""


def _run(tmp_path, program, args):
    src, exe = tmp_path / "shapes.hip", tmp_path / "shapes"
    src.write_text(program)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "snake-vk_amd", "csrc"), str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)] + [str(a) for a in args], check=True, capture_output=True, text=True).stdout
    return [[int(x) for x in line.split()] for line in out.splitlines()]


BATCH = r"""
#include <cstdio>
#include <cstdlib>
#include "snkpt_dev.h"
using namespace snkpt;
int main(int argc, char** argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        const uint32_t need = (uint32_t)atoi(argv[i]), lanes = (uint32_t)atoi(argv[i + 1]),
                       per_cu = (uint32_t)atoi(argv[i + 2]), n = (uint32_t)strtoul(argv[i + 3], nullptr, 10);
        with_stack(need, [&](auto s) {
            constexpr int S = decltype(s)::value;
            const TraceGrid g = batch_grid(S, lanes, per_cu, 256, n);
            printf("%u %u %u %d %d %u %u %u\n", lanes, per_cu, n, S, cu_waves(S), g.blocks, g.threads, g.lds);
        });
    }
    return 0;
}
"""


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_batch_grid(tmp_path):
    cus = 256
    cases = [(need, lanes, per_cu, n) for need in (6, 9, 11, 15, 30, 60) for lanes in (64, 128)
             for per_cu in (1, 4, 8, 16, 32, 64) for n in (1, 100, 38400, 500000, 15000000)]
    rows = _run(tmp_path, BATCH, [x for c in cases for x in c])
    assert len(rows) == len(cases)
    for lanes, per_cu, n, stack, cu_waves, blocks, threads, lds in rows:
        resident = cu_waves * 64 // lanes
        assert threads == lanes  # the block size asked for
        assert lds == 16 + stack * 8 * lanes and min(per_cu, resident) * lds <= 160 * 1024
        most = cus * min(per_cu, resident)
        assert 1 <= blocks <= most
        if n >= most * lanes:
            assert blocks == most  # the grid asked for
        else:
            assert blocks <= max(n // lanes + 1, cus)


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_trace_grid(tmp_path):
    cus = 256
    needs = [0, 6, 8, 9, 10, 11, 12, 13, 16, 17, 32, 33, 64]
    counts = [1, 7, 8, 9, 1000, 2048, 131073, 172800, 200000, 262144, 360448, 360449, 400000, 1 << 20, 2073600, (1 << 26) - 1]
    rows = _run(tmp_path, PROGRAM, [a for need in needs for n in counts for a in (need, n)])
    assert len(rows) == len(needs) * len(counts)
    for need, n, stack, cu_waves, widest, blocks, threads in rows:  # 22 waves' lanes per CU: the line
        waves = threads // 64
        assert stack >= need and threads % 64 == 0 and 1 <= waves <= widest and blocks >= 1
        # resident together: wave slots and 160 KB of LDS (16 B and 512 B per stack entry and wave)
        per_cu = -(-blocks // cus)
        assert per_cu * waves <= cu_waves
        assert per_cu * (16 + stack * 512 * waves) <= 160 * 1024
        if n <= cus * min(cu_waves, 22) * 64:
            # a lane for every ray; no more waves than the rays fill, once every CU has a block
            assert blocks * threads >= min(n, cus * (cu_waves // waves) * threads)
            assert blocks * threads <= max(n + threads, cus * threads), (need, n, blocks, threads)
            assert blocks <= max(1, (n + 7) // 8)
        else:
            assert blocks * waves >= cus * (cu_waves - waves + 1)  # the chip is filled
