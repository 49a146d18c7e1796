"""The library built for the CPU, for tests of what its kernels read and write.

``build()`` translates the HIP sources (dynamic and static LDS become allocations of their own, the few lines of inline
assembly become C++, the regions of a workspace get a gap between them that the address sanitizer watches; two, three and
five objectives only, which keeps the compile short) and compiles them with the runtime of ``tests/emulation``;
``run(specs)`` makes calls with it (``tests/emulation/calls.cpp``) and returns what it printed."""

import hashlib
import os
import re
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "emulation")
CXX = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and os.path.exists(c)), None)

_ASM = {
    'asm("v_addc_co_u32_e64 %0, %1, %2, %2, %3" : "=v"(r), "=s"(carry_out) : "v"(acc), "s"(mask));':
        "r = (acc << 1) | (uint32_t)((mask >> emu::cur->lane) & 1); (void)carry_out;",
    'asm("v_med3_i32 %0, %1, 0, 1" : "=v"(bit) : "v"(o));': "bit = (int)o > 0 ? 1u : 0u;",
    'asm("v_lshl_or_b32 %0, %1, 1, %2" : "=v"(r) : "v"(acc), "v"(bit));': "r = (acc << 1) | bit;",
    'asm("v_alignbit_b32 %0, %1, %2, 31" : "=v"(r) : "v"(acc), "v"(o));': "r = (acc << 1) | (o >> 31);",
    'asm volatile("s_waitcnt vmcnt(0)" ::: "memory");': "",
    '__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\\n\\ts_barrier" ::: "memory"); }':
        "#define lds_barrier() emu_sync()",
    'asm volatile("" : "+v"(tid));': ";",
    'asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));': "r = a > b ? a : b;",
    'asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));': "r = a < b ? a : b;",
    'asm volatile("global_load_dwordx4 %0, %1, off sc1\\n\\ts_waitcnt vmcnt(0)" : "=v"(r) : "v"(mine) : "memory");':
        "emu_load_pair(r, mine);",
}
_GAPS = """
#include <vector>
static thread_local bool emu_gaps_on = false;
static thread_local std::vector<std::pair<size_t, size_t>> emu_gaps;
static void emu_guard(uint8_t* base, size_t total, int batch, int64_t step) {
  for (int b = 0; b < batch; ++b) {
    uint8_t* const p = base + b * step;
    __asan_unpoison_memory_region(p, total);
    for (auto& g : emu_gaps) {
      const size_t a = (g.first + 7) / 8 * 8;
      if (a < g.second && g.second <= total) __asan_poison_memory_region(p + a, g.second - a);
    }
  }
}
"""


def _shared(line):
    """A line with a declaration of LDS, as a reference to memory of the workgroup."""
    m = re.match(r"(\s*)extern __shared__\s*(?:__attribute__\(\(aligned\(\d+\)\)\)\s*)?([\w ]+?)\s+(\w+)\[\];(.*)", line)
    if m:
        return f"{m[1]}{m[2]}* const {m[3]} = reinterpret_cast<{m[2]}*>(emu::dyn);{m[4]}"
    m = re.match(r"(\s*)__shared__\s*(?:__attribute__\(\(aligned\(\d+\)\)\)\s*)?(unsigned long long|\w+(?:<\w+>)?)\s+(.*?);(.*)", line)
    if not m:
        return line
    out, (indent, kind, names, rest) = "", m.groups()
    parts, depth = [""], 0
    for ch in names:
        depth += (ch in "[(<") - (ch in "])>")
        if ch == "," and depth == 0:
            parts.append("")
        else:
            parts[-1] += ch
    for part in parts:
        name, dims = re.match(r"\s*(\w+)(.*)", part).groups()
        out += (f"using emu_t_{name} = {kind}{dims}; static char emu_k_{name}; emu_t_{name}& {name} = "
                f"*reinterpret_cast<emu_t_{name}*>(emu::shared_at(&emu_k_{name}, sizeof(emu_t_{name}))); ")
    return indent + out + rest


def _replaced(text, old, new):
    assert old in text, f"the sources no longer hold {old!r}"
    return text.replace(old, new)


def _translate(name, text):
    text = "\n".join(_shared(line) for line in text.split("\n"))
    for old, new in _ASM.items():
        text = text.replace(old, new)
    text = re.sub(r"__attribute__\(\(amdgpu_waves_per_eu\(.*?\)\)\) void", "void", text)
    if "zero_words[" in text or "words[i] = 0u" in text:  # (one loop clears several regions and what lies between them)
        text = re.sub(r"(\w+)\[(\w)\] = 0u;", r"{ if (!__asan_address_is_poisoned(&\1[\2])) \1[\2] = 0u; }", text)
    text = re.sub(r"coherent_load\(&((?:a\.)?ctrl->err)\)", r"emu_error_word(&\1, kErrBarrierTimeout)", text)
    if name == "calibrate.hpp":
        text = re.sub(r"asm volatile\(.*?\);", ";", text, flags=re.S)
    if name == "peel_lds.hpp":
        a = text.index('asm volatile("global_load_dwordx4 %0, %2, off sc1')
        b = text.index(': "memory");', a) + len(': "memory");')
        where = re.search(r': "v"\((.*?)\)\s*: "memory"', text[a:b], re.S)[1]
        text = text[:a] + f"emu_load_pair(r0, {where}); emu_load_pair(r1, {where} + 2);" + text[b:]
    if name == "two_small.hpp":  # (a wave clears its counters and counts its items row by row in lockstep, without a barrier)
        text = _replaced(text, "cnt[wave * 256 + lane + 64 * i] = 0u;\n", "cnt[wave * 256 + lane + 64 * i] = 0u;\n  (void)emu_ballot(true);\n")
        text = _replaced(text, "reinterpret_cast<uint4*>(table)[2 * lane + 1] = zero;\n",
                         "reinterpret_cast<uint4*>(table)[2 * lane + 1] = zero;\n    (void)emu_ballot(true);\n")
        text = _replaced(text, "if (e - lane >= count) continue;", "if (e - lane >= count) continue; (void)emu_ballot(true);")
    if name == "api.hip":
        text = _replaced(text, "static size_t align_up(size_t v) { return (v + 255) / 256 * 256; }",
                         "static size_t align_up(size_t v) { if (!emu_gaps_on) return (v + 255) / 256 * 256; "
                         "const size_t e = (v + 255) / 256 * 256 + 256; emu_gaps.push_back({v, e}); return e; }")
        text = _replaced(text, "namespace evx {\n\nconstexpr int kMaxGrid", _GAPS + "namespace evx {\n\nconstexpr int kMaxGrid")
        text = _replaced(text, "  size_t o = 0;\n  // --- cleared", "  emu_gaps_on = true; emu_gaps.clear();\n  size_t o = 0;\n  // --- cleared")
        text = _replaced(text, "  L->wide_bytes = wide_workspace_need(n, m);",
                         "  emu_gaps_on = false; L->wide_bytes = wide_workspace_need(n, m); emu_gaps_on = true;")
        text = _replaced(text, "  L->total = o;\n  return true;", "  L->total = o;\n  emu_gaps_on = false;\n  return true;")
        text = _replaced(text, "  out->base = static_cast<uint8_t*>(ws);\n", "  out->base = static_cast<uint8_t*>(ws);\n  emu_guard(out->base, need, 1, 0);\n")
        text = _replaced(text, "    w.step = ws_step;\n", "    w.step = ws_step;\n    emu_guard(w.base, w.L.total, batch, ws_step);\n")
        text = re.sub(r"(?m)^\s*case (1|4|6|7|8|9|1\d): [^\n]*;\s*$", "", text)
    return text


def build():
    """The path of the program that makes the calls; compiled when a source has changed."""
    sources = [os.path.join(ROOT, "evox_amd", "csrc", f) for f in sorted(os.listdir(os.path.join(ROOT, "evox_amd", "csrc")))
               if f.endswith((".hpp", ".hip"))]
    mine = [os.path.join(HERE, f) for f in ("hip/hip_runtime.h", "emulator.cpp", "calls.cpp")]
    header = os.path.join(ROOT, "include", "evox_hip.h")
    digest = hashlib.sha256()
    for path in sources + mine + [header, os.path.abspath(__file__)]:
        with open(path, "rb") as f:
            digest.update(f.read())
    out = os.path.join(HERE, "build", digest.hexdigest()[:16])
    program = os.path.join(out, "calls")
    if os.path.exists(program):
        return program
    shutil.rmtree(os.path.join(HERE, "build"), ignore_errors=True)
    os.makedirs(os.path.join(out, "evox_amd", "csrc"))
    os.makedirs(os.path.join(out, "include"))
    shutil.copy(header, os.path.join(out, "include"))
    for path in sources:
        with open(path) as f:
            text = _translate(os.path.basename(path), f.read())
        with open(os.path.join(out, "evox_amd", "csrc", os.path.basename(path)), "w") as f:
            f.write(text)
    common = [CXX, "-std=c++17", "-g1", "-w", "-I", HERE, "-I", os.path.join(ROOT, "include")]
    guard = ["-fsanitize=address", "-mllvm", "-asan-stack=0", "-fno-omit-frame-pointer"]  # (the lanes' stacks are not its business)
    jobs = [
        common + guard + ["-O1", "-x", "c++", "-c", os.path.join(out, "evox_amd", "csrc", "api.hip"), "-o", os.path.join(out, "api.o")],
        common + ["-O2", "-c", mine[1], "-o", os.path.join(out, "emulator.o")],
        common + ["-O1", "-fsanitize=address", "-c", mine[2], "-o", os.path.join(out, "calls.o")],
    ]
    started = [subprocess.Popen(job, stderr=subprocess.PIPE, text=True) for job in jobs]
    for process in started:
        errors = process.communicate()[1]
        assert process.returncode == 0, errors[-4000:]
    checker = os.path.join(ROOT, "oracle", "libnd_oracle.so")
    if not os.path.exists(checker):
        subprocess.run(["make", "-C", os.path.join(ROOT, "oracle")], check=True)
    subprocess.run([CXX, "-fsanitize=address"] + [os.path.join(out, f) for f in ("api.o", "emulator.o", "calls.o")]
                   + [checker, "-Wl,-rpath," + os.path.dirname(checker), "-lpthread", "-o", program + ".tmp"], check=True)
    os.rename(program + ".tmp", program)
    return program


def run(specs, timeout=240, **environment):
    """What the calls printed; raises with the sanitizer's or the comparison's message when one of them failed."""
    done = subprocess.run([build()] + list(specs), env=dict(os.environ, **environment), capture_output=True, text=True, timeout=timeout)
    assert done.returncode == 0, done.stdout[-500:] + done.stderr[-6000:]
    return done.stdout + done.stderr
