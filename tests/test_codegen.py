"""What the kernels with hand-written waits and multiplies rest on, checked in the code that the compiler made of them.

An asm statement that loads or multiplies hides its latency from the compiler, which takes the result as written at once: it could copy a
register between the load and its wait, or a sum behind a multiply that is still on its way, and no source line would show it.  The check follows every
path through the disassembly of the kernels built here and finds such a use, whatever compiler built them."""
import functools
import re
import subprocess
from pathlib import Path

import pytest

from orinfer_amd import build, lib

LLVM = Path(build.hipcc()).resolve().parents[1]
OBJDUMP = next((p for p in (LLVM / "llvm/bin/llvm-objdump", LLVM / "lib/llvm/bin/llvm-objdump", Path("/opt/rocm/llvm/bin/llvm-objdump")) if p.exists()), None)
FAR = 64  # wait states, or younger requests: as good as any number
RESULT_WAIT = 8  # wait states that the compiler itself keeps between v_mfma_i32_16x16x64_i8 and another access to its sum


def parse_registers(text):
    """VGPRs as their numbers, accumulation registers from 1000 on."""
    found = []
    for kind, one, low, high in re.findall(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        numbers = range(int(one), int(one) + 1) if one else range(int(low), int(high) + 1)
        found.extend(n + (1000 if kind == "a" else 0) for n in numbers)
    return tuple(found)


class Instruction:
    def __init__(self, text):
        self.text = text
        self.name, _, operands = text.partition(" ")
        first = parse_registers(operands.partition(",")[0])
        self.all = parse_registers(operands)
        if self.name == "v_mad_u64_u32":  # (made of 32-bit sums too: the addend's upper half is then any register, and nobody reads the result's)
            self.all = self.all[:-1]
        self.multiply = self.name.startswith("v_mfma")
        self.sum = first if self.multiply else ()
        self.memory = self.name.startswith(("global_", "buffer_", "flat_", "scratch_"))
        self.wide = self.name in ("global_load_dwordx2", "global_load_dwordx4")
        self.loads = first if self.wide or self.name in ("global_load_dword", "global_load_ushort") else ()
        self.lds = self.name.startswith("ds_")
        self.reads = first if self.name.startswith(("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle")) or "_rtn_" in self.name and self.lds else ()
        self.move = self.name.startswith(("v_mov", "v_accvgpr", "v_swap", "scratch_"))
        counted = re.search(r"vmcnt\((\d+)\)", text) if self.name == "s_waitcnt" else None
        self.younger = int(counted.group(1)) if counted else None
        counted = re.search(r"lgkmcnt\((\d+)\)", text) if self.name == "s_waitcnt" else None
        self.younger_lds = int(counted.group(1)) if counted else None
        self.states = 1 + (int(operands) if self.name == "s_nop" else 0)


def kernels(listing):
    """(name, [(address, Instruction)], {address of a branch: its target}) of every kernel in a disassembly."""
    name, code, targets, base = None, [], {}, 0
    known = {}
    for line in listing.splitlines():
        header = re.match(r"^([0-9a-f]+) <(.*)>:", line)
        if header:
            if code:
                yield name, code, targets
            name, code, targets, base = header.group(2), [], {}, int(header.group(1), 16)
            continue
        text, _, comment = line.partition("//")
        text = " ".join(text.split())
        if not text or not comment:
            continue
        address = int(comment.split(":")[0], 16)
        target = re.search(r"<.*?(?:\+0x([0-9a-f]+))?>\s*$", comment)
        if text.startswith(("s_cbranch", "s_branch")):
            targets[address] = base + int(target.group(1) or "0", 16)
            text = text.split()[0]
        code.append((address, known.setdefault(text, Instruction(text))))
    if code:
        yield name, code, targets


def faults(code, targets, by_condition=False):
    """Uses of a register whose load, LDS read or multiply may not have ended, over all paths; of 8 and 16 bytes in flight from memory, moves only.  (The waits for those hang
    together with their requests by uniform conditions and loop counts, which a walk over all paths does not know.  A wave's LDS operations end in order; scalar loads, which share
    their counter, can only make a wait longer, so they count for nothing.  by_condition: moves only for these too, in kernels
    whose reads and waits are both behind the same uniform condition.)"""
    index = {address: i for i, (address, _) in enumerate(code)}
    starts = {0} | {index[t] for t in targets.values()} | {index[a] + 1 for a in targets}
    found, seen, work = set(), {}, [(0, ({}, {}, {}))]
    while work:
        i, state = work.pop()
        if i in seen:  # the shortest way to every register's last event
            merged = tuple({r: min(old.get(r, FAR), new.get(r, FAR)) for r in {*old, *new}} for old, new in zip(seen[i], state))
            if merged == seen[i]:
                continue
            state = merged
        seen[i] = state
        loaded, multiplied, read = dict(state[0]), state[1], state[2]  # younger requests, by register and width; wait states since; younger LDS operations
        while True:
            address, ins = code[i]
            for r in ins.all:
                if (r, False) in loaded or (ins.move and (r, True) in loaded):
                    found.add(f"{ins.text}: register {r} is on its way")
                if r in read and (ins.move or not by_condition):
                    found.add(f"{ins.text}: register {r} is on its way from LDS")
                if r in multiplied and not ins.multiply:
                    found.add(f"{ins.text}: register {r} is a sum of {multiplied[r]} wait states ago")
            multiplied = {r: n + ins.states for r, n in multiplied.items() if n + ins.states < RESULT_WAIT}
            if ins.multiply:
                multiplied.update(dict.fromkeys(ins.sum, 0))
            if ins.memory:
                loaded = {r: n + 1 for r, n in loaded.items()}
                for r in ins.loads:
                    loaded.pop((r, not ins.wide), None)
                    loaded[r, ins.wide] = 0
            if ins.lds:
                read = {r: n + 1 for r, n in read.items() if r not in ins.reads}
                read.update(dict.fromkeys(ins.reads, 0))
            if ins.younger_lds is not None:
                read = {r: n for r, n in read.items() if n < ins.younger_lds}
            if ins.younger is not None:
                loaded = {r: n for r, n in loaded.items() if n < ins.younger}
            if ins.name == "s_endpgm":
                break
            if address in targets:
                work.append((index[targets[address]], (loaded, multiplied, read)))
                if ins.name == "s_branch":
                    break
            i += 1
            if i == len(code):
                break
            if i in starts:
                work.append((i, (loaded, multiplied, read)))
                break
    return found


SCALAR_WAIT = 2  # wait states that the compiler itself keeps between a vector instruction that writes a scalar register and one that reads it
TO_MEMORY_WAIT = 5  # and before a memory instruction that reads it


def scalar_registers(text):
    found = set()
    for name, one, low, high in re.findall(r"\b(?:(vcc)\b|s(\d+)\b|s\[(\d+):(\d+)\])", text):
        found |= {"vcc"} if name else {int(one)} if one else set(range(int(low), int(high) + 1))
    return found


@functools.lru_cache(maxsize=None)
def scalars_of(text):
    """(scalar registers that a vector instruction writes, those that it or a memory instruction reads)."""
    name, _, operands = text.partition(" ")
    if name.startswith(("global_", "buffer_", "flat_", "scratch_")):
        return set(), scalar_registers(operands)
    if not name.startswith("v_"):
        return set(), set()
    parts = re.split(r",(?![^\[]*\])", operands.replace("vcc_lo", "vcc").replace("vcc_hi", "vcc"))
    results = 2 if re.match("v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[ui]64", name) else 1
    writes, reads = scalar_registers(",".join(parts[:results])), scalar_registers(",".join(parts[results:]))
    if re.match("v_div_fmas|v_cndmask_b32_(e32|dpp|sdwa)", name):
        reads |= {"vcc"}
    return writes, reads


def early_scalars(code, targets):
    """Vector and memory instructions that read a scalar register too soon behind the vector instruction that writes it, on any path.  The compiler spaces its own instructions and
    does not look into asm statements."""
    index, found = {address: i for i, (address, _) in enumerate(code)}, set()
    for start, (_, writer) in enumerate(code):
        written = scalars_of(writer.text)[0]
        if not written:
            continue
        following = lambda i: ([index[targets[code[i][0]]]] if code[i][0] in targets else []) + ([i + 1] if code[i][1].name not in ("s_branch", "s_endpgm") and i + 1 < len(code) else [])
        work = [(i, 0, written) for i in following(start)]
        while work:
            i, states, left = work.pop()
            ins = code[i][1]
            writes, reads = scalars_of(ins.text)
            if reads & left and states < (TO_MEMORY_WAIT if ins.memory else SCALAR_WAIT):
                found.add(f"{ins.text}: {states} wait states behind {writer.text}")
            left = left - writes - (scalar_registers(ins.text.partition(" ")[2].partition(",")[0]) if ins.name.startswith("s_") else set())
            states += ins.states
            if left and states < TO_MEMORY_WAIT:
                work.extend((next_one, states, left) for next_one in following(i))
    return found


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    """The code objects in the library, disassembled: {kernel: (code, targets)}."""
    folder = tmp_path_factory.mktemp("code")
    (folder / "lib.so").write_bytes(Path(lib.LIBRARY_PATH).read_bytes())
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    out = {}
    for part in sorted(folder.glob("*gfx950*")):
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", part.name], cwd=folder, check=True, capture_output=True, text=True).stdout
        out.update({name: (code, targets) for name, code, targets in kernels(listing)})
    return out


@pytest.mark.parametrize("family, count", [("panel_kernel", 60), ("runs_kernel", 50), ("grouped_bulk_kernel", 8), ("gemm_mid_kernel", 2), ("gemm_big_persistent_kernel", 4)])
def test_nothing_touches_a_register_that_is_on_its_way(built, family, count):
    chosen = {name: code for name, code in built.items() if family in name}
    assert len(chosen) >= count
    for name, (code, targets) in chosen.items():
        by_condition = re.search("panel_kernel.*Lb0E", name) is not None  # (waves that share the last block of a run unevenly)
        assert not (problems := faults(code, targets, by_condition)), (name, sorted(problems)[:5])


@pytest.mark.parametrize("lines, found", [
    (["ds_read_b128 v[0:3], v9", "v_mov_b32_e32 v20, v0", "s_waitcnt lgkmcnt(0)"], True),
    (["ds_read_b128 v[0:3], v9", "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v20, v0"], False),
    (["ds_read_b128 v[0:3], v9", "ds_read_b64 v[4:5], v9", "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v20, v0"], False),
    (["ds_read_b128 v[0:3], v9", "ds_read_b64 v[4:5], v9", "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v20, v5"], True),
    (["ds_read_b128 v[0:3], v9", "ds_write_b64 v9, v[4:5]", "s_waitcnt lgkmcnt(1)", "v_add_u32_e32 v20, v3, v3"], False),
    (["ds_read_b128 v[0:3], v9", "s_load_dword s0, s[2:3], 0x0", "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v20, v0"], True),  # a scalar load may end first
    (["ds_read_b128 v[0:3], v9", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v2, v20"], True),                                    # another counter; a write
    (["global_load_dwordx4 v[0:3], v9, s[2:3]", "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v20, v0"], True),
    (["v_mfma_i32_16x16x64_i8 v[0:3], v[4:7], v[8:11], v[0:3]", "s_nop 5", "v_mov_b32_e32 v20, v0"], True),
    (["v_mfma_i32_16x16x64_i8 v[0:3], v[4:7], v[8:11], v[0:3]", "s_nop 7", "v_mov_b32_e32 v20, v0"], False)])
def test_the_walk_finds_a_use_in_front_of_its_wait(lines, found):
    code = [(4 * i, Instruction(text)) for i, text in enumerate(lines + ["s_endpgm"])]
    assert bool(faults(code, {})) == bool(faults(code, {}, True)) == found


def test_no_instruction_reads_a_scalar_register_too_soon_behind_a_vector_instruction(built):
    assert len(built) > 400
    for name, (code, targets) in built.items():
        assert not (problems := early_scalars(code, targets)), (name, sorted(problems)[:5])


@pytest.mark.parametrize("lines, found", [
    (["v_subb_co_u32_e64 v0, vcc, v1, v2, s[0:1]", "v_addc_co_u32_e32 v3, vcc, 0, v3, vcc"], True),
    (["v_subb_co_u32_e64 v0, vcc, v1, v2, s[0:1]", "s_nop 1", "v_addc_co_u32_e32 v3, vcc, 0, v3, vcc"], False),
    (["v_subb_co_u32_e64 v0, vcc, v1, v2, s[0:1]", "s_nop 0", "v_addc_co_u32_e32 v3, vcc, 0, v3, vcc"], True),
    (["v_subb_co_u32_e64 v0, s[4:5], v1, v2, s[0:1]", "v_mov_b32_e32 v9, v8", "v_addc_co_u32_e64 v3, s[4:5], 0, v3, s[4:5]"], True),
    (["v_subb_co_u32_e64 v0, s[4:5], v1, v2, s[0:1]", "v_subb_co_u32_e64 v0, s[6:7], v1, v4, s[2:3]", "v_mov_b32_e32 v9, v8", "v_addc_co_u32_e64 v3, s[4:5], 0, v3, s[4:5]"], False),
    (["v_cmp_lt_u32_e64 s[4:5], v1, v2", "s_and_b64 s[4:5], s[4:5], s[6:7]", "v_cndmask_b32_e64 v0, v0, 0, s[4:5]"], False),  # a scalar instruction's result
    (["v_cmp_lt_u32_e32 vcc, v1, v2", "v_cndmask_b32_e32 v0, v0, v3, vcc"], True),
    (["v_readfirstlane_b32 s4, v1", "s_nop 1", "v_add_u32_e32 v0, s4, v0"], False),
    (["v_readfirstlane_b32 s4, v1", "s_nop 3", "global_load_dword v0, v1, s[4:5]"], True),
    (["v_readfirstlane_b32 s4, v1", "s_nop 4", "global_load_dword v0, v1, s[4:5]"], False)])
def test_the_walk_finds_a_scalar_register_that_is_read_too_soon(lines, found):
    code = [(4 * i, Instruction(text)) for i, text in enumerate(lines + ["s_endpgm"])]
    assert bool(early_scalars(code, {})) == found
    assert bool(early_scalars([(0, Instruction("s_branch"))] + [(4 * i + 4, Instruction(text)) for i, text in enumerate(lines + ["s_endpgm"])], {0: 4})) == found


def test_the_walk_follows_a_read_around_a_loop():
    """A fragment read at the end of a step for the next one, whose wait stands in front of the multiplies: a copy at the loop's head is in front of it."""
    step = ["s_waitcnt lgkmcnt(0)", "v_mfma_i32_16x16x64_i8 v[16:19], v[0:3], v[0:3], v[16:19]", "ds_read_b128 v[0:3], v9", "s_cbranch_scc1", "s_endpgm"]
    for lines, found in ((step, False), (["v_mov_b32_e32 v20, v0"] + step, True)):
        code = [(4 * i, Instruction(text)) for i, text in enumerate(lines)]
        assert bool(faults(code, {4 * lines.index("s_cbranch_scc1"): 0})) == found


def test_sums_of_the_panel_kernel_stay_where_they_are(built):
    """Its multiplies are asm statements on every side of a branch: no register moves between the first and the last, and only multiplies name the sums."""
    for name, (code, _) in built.items():
        if "panel_kernel" not in name:
            continue
        at = [i for i, (_, ins) in enumerate(code) if ins.multiply]
        sums = {r for i in at for r in code[i][1].sum}
        for _, ins in code[at[0]:at[-1]]:
            assert ins.multiply or not sums & set(ins.all), (name, ins.text)
            assert not ins.name.startswith(("v_mov", "v_accvgpr", "v_swap", "scratch_")), (name, ins.text)


def test_requests_that_share_an_lds_base_keep_it(built):
    """Kernels with a request that sets no m0 of its own write m0 nowhere but in front of one that does."""
    families = 0
    for name, (code, _) in built.items():
        if not ("grouped_bulk_kernel" in name or "panel_kernelILi1" in name or "runs_kernelILi0" in name):
            continue
        texts, families = [ins.text for _, ins in code], families + 1
        for i, text in enumerate(texts):
            if re.search(r"\bm0\b", text):
                assert text.startswith("s_mov_b32 m0, ") and texts[i + 1] == "s_nop 0" and texts[i + 2].startswith("global_load_lds_dwordx4"), (name, texts[i:i + 3])
    assert families >= 4 + 30 + 32


def test_a_request_does_not_hide_the_lds_base_of_a_builtin(tmp_path):
    """request_16 between two direct_load_16 to one place: the second sets its base again."""
    source = tmp_path / "both.hip"
    source.write_text('''#include "lds_asm.h"
using namespace orx::lds_asm;
extern "C" __global__ void both(const uint8_t* a, const uint8_t* b, int* out) {
    __shared__ __align__(16) uint8_t first[1024], second[1024];
    direct_load_16(a + threadIdx.x * 16, first);
    request_16<REQUEST>(threadIdx.x * 16, b, lds_address_of(second));
    direct_load_16(a + threadIdx.x * 16 + 4096, first);
    __syncthreads();
    out[threadIdx.x] = first[threadIdx.x] + second[threadIdx.x];
}
''')
    done = subprocess.run([build.hipcc(), *build.FLAGS, "-Werror=inline-asm", f"-I{build.CSRC}", "-DREQUEST=0", "--cuda-device-only", "-S", str(source), "-o", "-"],
                          capture_output=True, text=True, check=True)
    order = [line.split()[0] for line in done.stdout.splitlines() if re.match(r"\s+(s_mov_b32 m0|global_load_lds)", line)]
    assert order == ["s_mov_b32", "global_load_lds_dwordx4"] * 3
