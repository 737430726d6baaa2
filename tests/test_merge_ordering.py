"""The split-KV merge inside the forward launch (csrc/intfa_splitkv.h) reads partials that other workgroups wrote.  What the compiler is given
must hold the order: stores of partials at agent scope, a wait for them, the ticket's atomic addition, an acquire fence, loads of partials
at agent scope.  Compiles the two arrival functions, as the kernels call them and each between a store and a load of a partial, to the compiler's
intermediate form."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "intfa_splitkv.h"
using namespace intfa;
__global__ void arrive_workgroup(const KParams p, float* out) {
    __shared__ __attribute__((aligned(16))) char smem[64];
    const KernargPtr pe = kernarg_block();
    const SplitPartials part(pe, 128, 0);
    part.put_lse(threadIdx.x, 1.f);
    if (!splitkv_last_arrival(pe, smem, blockIdx.x)) return;
    out[threadIdx.x] = part.get_lse(threadIdx.x);
}
__global__ void arrive_wave(const KParams p, float* out) {
    const KernargPtr pe = kernarg_block();
    const SplitPartials part(pe, 128, 0);
    part.put_lse(threadIdx.x, 1.f);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!splitkv_last_arrival_wave(pe, blockIdx.x)) return;
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


# The arrival's answer lies in the first bytes of the workgroup's LDS and is read without a barrier behind it, so a wave that is in the merge
# already must not write there: every rule of splitkv_merge_rows and splitkv_merge_many for a place in LDS, at every head_dim and both
# numbers of waves.
MERGE_SOURCE = """
#include "intfa_splitkv.h"
using namespace intfa;
template <int D, int WAVES> __device__ __forceinline__ void arrive_and_merge(char* smem, int nrows) {
    const KernargPtr p = kernarg_block();
    if (splitkv_last_arrival(p, smem, blockIdx.x)) splitkv_merge_rows<D, 0, WAVES>(p, smem, 0, blockIdx.x, 0, nrows);
}
#define MERGE(D, W) __global__ void merge_d##D##_w##W(const KParams p, int nrows) { \\
    __shared__ __attribute__((aligned(16))) char smem[kMergeLds]; arrive_and_merge<D, W>(smem, nrows); }
MERGE(64, 4) MERGE(64, 8) MERGE(128, 4) MERGE(128, 8) MERGE(256, 4) MERGE(256, 8)
"""


def lowest_offset(expr, defs):
    """The smallest value that an address (bytes from the LDS array) or an index of the compiler's intermediate form can take.  What is not
    arithmetic is a thread's, wave's or loop's number or a masked one: not negative."""
    expr = expr.strip()
    if re.fullmatch(r"-?\d+", expr):
        return int(expr)
    m = re.fullmatch(r"getelementptr (?:inbounds |nuw |nusw )*\((.*?), ptr addrspace\(3\) (@\w+), i32 (\d+)\)", expr)
    if m:
        return {"i8": 1, "i32": 4, "float": 4, "<4 x float>": 16}[m.group(1)] * int(m.group(3))
    if expr.startswith("@"):
        return 0
    d = defs.get(expr, "")
    m = re.match(r"getelementptr (?:inbounds |nuw |nusw )*(i8|i32|float|<4 x float>), ptr addrspace\(3\) (%\S+|@\w+|getelementptr .*\)), i32 (\S+)$", d)
    if m:
        return lowest_offset(m.group(2), defs) + {"i8": 1, "i32": 4, "float": 4, "<4 x float>": 16}[m.group(1)] * lowest_offset(m.group(3), defs)
    m = re.match(r"(add|or|shl|mul) (?:nuw |nsw |disjoint )*i32 (\S+), (\S+)$", d)
    if m:
        a, b = (lowest_offset(x, defs) for x in m.group(2, 3))
        return {"add": a + b, "or": max(a, b), "shl": a << max(b, 0), "mul": a * b}[m.group(1)]
    return 0


def test_the_merge_writes_no_byte_of_the_arrivals_answer(tmp_path):
    src, out = tmp_path / "merges.hip", tmp_path / "merges.ll"
    src.write_text(MERGE_SOURCE)
    r = subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-I", os.path.join(ROOT, "int-flashattention_amd", "csrc"), "--offload-device-only", "-emit-llvm", "-S", str(src),
                        "-o", str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    bodies = re.findall(r"^define [^\n]*@_Z\d+(merge_d\d+_w\d)\w*\([^\n]*\n(.*?)^}", out.read_text(), re.S | re.M)
    assert len(bodies) == 6
    for name, body in bodies:
        defs = dict(re.findall(r"^  (%\S+) = (.*?)(?:, !.*)?$", body, re.M))
        stores = re.findall(r"^  store (i32|float|<4 x float>) (?:<[^>]*>|[^,]*), ptr addrspace\(3\) (.*?), align", body, re.M)
        assert len(stores) == len(re.findall(r"^  store .*addrspace\(3\)", body, re.M)) and len(stores) >= 6, name
        answer = [a for t, a in stores if t == "i32"]
        assert len(answer) == 1 and lowest_offset(answer[0], defs) == 0, name
        for t, a in stores:
            if t != "i32":
                assert lowest_offset(a, defs) >= 4, f"{name}: a {t} of the merge may lie on the arrival's answer ({a})"
