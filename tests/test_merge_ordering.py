"""The split-KV merge inside the forward launch (csrc/intfa_splitkv.h) reads partials that other workgroups wrote.  What the compiler is given
must hold the order: stores of partials at agent scope, a wait for them, the ticket's atomic addition, an acquire fence, loads of partials
at agent scope.  Compiles the two arrival functions, each between a store and a load of a partial, to the compiler's intermediate form."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "intfa_splitkv.h"
using namespace intfa;
__global__ void arrive_workgroup(const KParams p, float* out) {
    __shared__ __attribute__((aligned(16))) char smem[64];
    const SplitPartials part(&p, 128, 0);
    part.put_lse(threadIdx.x, 1.f);
    if (!splitkv_last_arrival(p, smem, blockIdx.x)) return;
    out[threadIdx.x] = part.get_lse(threadIdx.x);
}
__global__ void arrive_wave(const KParams p, float* out) {
    const SplitPartials part(&p, 128, 0);
    part.put_lse(threadIdx.x, 1.f);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!splitkv_last_arrival_wave(&p, blockIdx.x)) return;
    out[threadIdx.x] = part.get_lse(threadIdx.x);
}
"""


def test_the_merge_reads_behind_a_fence_and_arrives_behind_its_stores(tmp_path):
    src = tmp_path / "arrivals.hip"
    src.write_text(SOURCE)
    out = tmp_path / "arrivals.ll"
    r = subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-I", os.path.join(ROOT, "int-flashattention_amd", "csrc"), "--offload-device-only", "-emit-llvm", "-S", str(src),
                        "-o", str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    bodies = re.findall(r"^define [^\n]*@_Z\d+(arrive_workgroup|arrive_wave)\w*\([^\n]*\n(.*?)^}", out.read_text(), re.S | re.M)
    assert {n for n, _ in bodies} == {"arrive_workgroup", "arrive_wave"}
    agent = r"i32 0, i32 16\)"                       # offset, cache policy: sc1
    for name, body in bodies:
        lines, pos = body.splitlines(), 0
        for what in (r"call void @llvm\.amdgcn\.raw\.ptr\.buffer\.store.*" + agent, r"asm sideeffect \"s_waitcnt vmcnt\(0\)\".*~\{memory\}",
                     r"atomicrmw add .*syncscope\(\"agent[^\"]*\"\) monotonic", r"fence (syncscope\(\"[a-z-]+\"\) )?acquire$",
                     r"@llvm\.amdgcn\.raw\.ptr\.buffer\.load.*" + agent):
            pos = next((i + 1 for i in range(pos, len(lines)) if re.search(what, lines[i])), None)
            assert pos is not None, f"{name}: no `{what}` in its place"
        first_load = next(i for i, line in enumerate(lines) if "raw.ptr.buffer.load" in line)
        assert first_load + 1 == pos, f"{name}: a partial is read ahead of the fence"
