"""What the compiler made of the kernels, read from the built library: its metadata and its instructions."""
import os
import re
import subprocess

import pytest

from bytetransformer_amd import build

LLVM = os.path.join(build.ROCM, "llvm", "bin")
KERNELS = os.path.join(build.LIB, "libbt_hip.so")
pytestmark = pytest.mark.skipif(not os.path.exists(KERNELS), reason="the kernels have not been built")


def _tool(name, *args):
    return subprocess.run([os.path.join(LLVM, name)] + list(args), check=True, stdout=subprocess.PIPE, text=True).stdout


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The library's gfx950 code objects, one per source file, as files."""
    tmp = tmp_path_factory.mktemp("code")
    fat = str(tmp / "fat")
    _tool("llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, KERNELS, str(tmp / "rest"))
    data = open(fat, "rb").read()
    # one bundle per source file, each starting with this magic
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)] + [len(data)]
    files = []
    for i, (at, end) in enumerate(zip(starts, starts[1:])):
        bundle, code = str(tmp / ("bundle%d" % i)), str(tmp / ("code%d" % i))
        with open(bundle, "wb") as f:
            f.write(data[at:end])
        _tool("clang-offload-bundler", "--unbundle", "--type=o", "--input=" + bundle, "--output=" + code,
              "--targets=hipv4-amdgcn-amd-amdhsa--gfx950")
        files.append(code)
    assert len(files) == len(build.KERNEL_SOURCES)
    return files


def test_no_kernel_spills(code_objects):
    """A kernel that does not fit its registers pays for it in every tile (the wide attention kernel under mask
    and bias took 97 us in place of 75): none has spilled registers or scratch memory."""
    kernels = {}
    for code in code_objects:
        for block in re.split(r"\n  - \.agpr_count", _tool("llvm-readelf", "--notes", code))[1:]:
            keys = dict(re.findall(r"\.(vgpr_spill_count|private_segment_fixed_size): +(\d+)", block))
            kernels[re.search(r"\.name: +(\S+)", block).group(1)] = {k: int(v) for k, v in keys.items()}
    assert sum("attention_grouped_kernel" in k for k in kernels) >= 12 and len(kernels) > 100
    bad = {k: v for k, v in kernels.items() if v["vgpr_spill_count"] or v["private_segment_fixed_size"]}
    assert not bad, bad


def test_products_bring_few_argument_bytes(code_objects):
    """Every argument byte costs the host, most of it beyond 80 (0.5 us a launch): only launches that count mask rows
    bring their fields."""
    sizes = {}
    for code in code_objects:
        for block in re.split(r"\n  - \.agpr_count", _tool("llvm-readelf", "--notes", code))[1:]:
            name = re.search(r"\.name: +(\S+)", block).group(1)
            m = re.search(r"gemm_(?:flat_|wave_k_|few_rows_)?kernelI(.*)EEv", name)
            if m and "f32" not in name:
                ints = re.findall(r"L[ib](\d+)E", m.group(1) + "E")
                mask = {"gemm_kernel": ints[8:9], "gemm_flat": ints[8:9], "gemm_wave": ints[2:3]}.get(
                    re.search(r"gemm_[a-z]+", name).group(0), ["0"])[0]
                sizes.setdefault(mask != "0", set()).add(int(re.search(r"\.kernarg_segment_size: +(\d+)", block).group(1)))
    assert max(sizes[False]) <= 80 and max(sizes[True]) <= 112, sizes


def test_the_streaming_attention_brings_few_argument_bytes(code_objects):
    """The same for the 64-wide attention: 176 bytes as one struct before its first arguments came in registers."""
    sizes = {}
    for code in code_objects:
        for block in re.split(r"\n  - \.agpr_count", _tool("llvm-readelf", "--notes", code))[1:]:
            m = re.search(r"\.name: +\S*attention_grouped_kernelILi\dELi(\d)E", block)
            if m:
                terms = int(m.group(1)) in (1, 2, 3)
                sizes.setdefault(terms, set()).add(int(re.search(r"\.kernarg_segment_size: +(\d+)", block).group(1)))
    assert max(sizes[False]) <= 128 and max(sizes[True]) <= 152, sizes


# Wait states between a matrix instruction and the first other use of its result, which the hardware does not enforce:
# passes + 4 on the XDL units (16-bit operands), passes + 2 on the others.
RESULT_WAIT = {"v_mfma_f32_32x32x2_f32": 16 + 2, "v_mfma_f32_16x16x4_f32": 8 + 2, "v_mfma_f32_32x32x16_f16": 8 + 4,
               "v_mfma_f32_32x32x16_bf16": 8 + 4, "v_mfma_f32_16x16x32_f16": 4 + 4}


def _registers(operand):
    m = re.match(r"-?\|?([va])(?:(\d+)|\[(\d+):(\d+)\])\|?$", operand)
    if not m:
        return frozenset()
    first, last = (m.group(2), m.group(2)) if m.group(2) else (m.group(3), m.group(4))
    return frozenset((m.group(1), i) for i in range(int(first), int(last) + 1))


def _functions(code):
    """(name, [(opcode, operands)], [successors]) of every function of a code object."""
    name, lines = None, []
    for line in _tool("llvm-objdump", "-d", "--no-show-raw-insn", code).split("\n") + ["0 <end>:"]:
        head = re.match(r"[0-9a-f]+ <(\S+)>:$", line)
        if head:
            if lines:
                at = {address: i for i, (address, _, _, _) in enumerate(lines)}
                after = []
                for i, (_, op, _, target) in enumerate(lines):
                    jump = [at[lines[0][0] + target]] if target is not None else []
                    goes_on = op not in ("s_branch", "s_endpgm") and i + 1 < len(lines)
                    after.append(jump + ([i + 1] if goes_on else []))
                yield name, [(op, operands) for _, op, operands, _ in lines], after
            name, lines = head.group(1), []
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(?:.*<\S+?\+0x([0-9a-f]+)>)?", line)
        if m:
            op, text, address, target = m.groups()
            jumps = op.startswith(("s_branch", "s_cbranch"))
            lines.append((int(address, 16), op, [t for t in re.split(r",\s*|\s+", text) if t],
                          int(target, 16) if jumps and target else None))


def _early_uses(name, code, after):
    found = []
    used = [[_registers(t) for t in operands] for _, operands in code]
    for i, (op, operands) in enumerate(code):
        if not op.startswith("v_mfma"):
            continue
        result, need, best, todo = used[i][0], RESULT_WAIT[op], {}, [(j, 0) for j in after[i]]
        while todo:
            j, waited = todo.pop()
            if waited >= need or best.get(j, need) <= waited:
                continue
            best[j] = waited
            other = code[j][0]
            registers = used[j]
            if other.startswith("v_mfma"):
                registers = used[j][1:3]     # (the accumulator of a chain is forwarded)
            elif re.match(r"(ds_read|global_load|buffer_load)", other):
                registers = used[j][1:]      # (what a load returns arrives long after)
            if any(r & result for r in registers):
                found.append("%s: %s %s, then %s %s after %d of %d wait states" % (
                    name, op, ", ".join(operands), other, ", ".join(code[j][1]), waited, need))
                continue
            if other.startswith("v_mfma") and used[j][0] >= result:
                continue                     # overwritten by the next of the chain, which is looked at itself
            step = int(code[j][1][0], 0) + 1 if other == "s_nop" else 1
            todo += [(k, waited + step) for k in after[j]]
    return found


def test_no_kernel_reads_a_matrix_result_early(code_objects):
    """Over every path through every kernel, loops included. (The float attention's last read came 11 wait states
    early: its last columns were wrong at head sizes 96 and 128.)"""
    early, matrix = [], 0
    for code in code_objects:
        for name, instructions, after in _functions(code):
            matrix += sum(op.startswith("v_mfma") for op, _ in instructions)
            early += _early_uses(name, instructions, after)
    assert matrix > 1000
    assert not early, early


def test_the_compiler_knows_every_store():
    """Assembly that stores is nothing to the compiler: it neither waits for the matrix instruction whose result goes
    out nor keeps the store in order with other accesses to the same memory."""
    folder = os.path.join(build.CSRC, "kernels")
    hidden = [(f, text) for f in sorted(os.listdir(folder)) if f.endswith((".h", ".hip"))
              for text in re.findall(r"\basm(?:\s+volatile)?\s*\(([^;]*);", open(os.path.join(folder, f)).read())
              if re.search(r"(global|buffer|flat|scratch)_(store|atomic)|ds_(write|add|max)", text)]
    assert not hidden, hidden


LOAD = re.compile(r"(ds_read|ds_bpermute|ds_permute|ds_swizzle|global_load|buffer_load|flat_load|scratch_load)")
COUNTED = {"lgkmcnt": re.compile(r"ds_"), "vmcnt": re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)")}


def _touched_in_flight(name, code, after):
    """Loads whose destination another instruction reads or writes before a wait has made sure of their return. (They
    return in order, so `s_waitcnt counter(n)` has waited for a load with n or more counted operations behind it.)"""
    found = []
    used = [frozenset().union(*[_registers(t) for t in operands]) if operands else frozenset() for _, operands in code]
    waits = []
    for op, operands in code:
        # (a function waits for everything before it does anything else)
        text = "vmcnt(0) lgkmcnt(0)" if op == "s_swappc_b64" else " ".join(operands)
        waits.append({c: int(n) for c, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", text)} if op in ("s_waitcnt", "s_swappc_b64") else {})
    for i, (op, operands) in enumerate(code):
        if not LOAD.match(op) or "lds" in operands or "_lds_" in op:
            continue                                     # (no register waits for a load into LDS)
        counter = "lgkmcnt" if op.startswith("ds_") else "vmcnt"
        result, least, todo = _registers(operands[0]), {}, [(j, 0) for j in after[i]]
        while todo:
            j, behind = todo.pop()
            if least.get(j, 1 << 30) <= behind:
                continue
            least[j] = behind
            if waits[j].get(counter, 1 << 30) <= behind:
                continue
            other, its = code[j]
            if used[j] & result:
                # (another load of the kind into the same registers returns after this one)
                if not (LOAD.match(other) and COUNTED[counter].match(other) and _registers(its[0]) >= result and
                        not any(_registers(t) & result for t in its[1:])):
                    found.append("%s: %s %s in flight at %s %s" % (name, op, ", ".join(operands), other, ", ".join(its)))
                continue
            behind = min(behind + bool(COUNTED[counter].match(other)), 64)
            todo += [(k, behind) for k in after[j]]
    return found


def test_no_kernel_touches_a_register_that_a_load_is_about_to_write(code_objects):
    """Over every path through every kernel. (The cache warm-up left its loads in flight into a register that the
    next turn of the loop computed an address in: an illegal access, once in a long while.)"""
    touched, loads = [], 0
    for code in code_objects:
        for name, instructions, after in _functions(code):
            loads += sum(bool(LOAD.match(op)) for op, _ in instructions)
            touched += _touched_in_flight(name, instructions, after)
    assert loads > 5000
    assert not touched, (len(touched), touched[:20])


def test_the_search_for_loads_in_flight_finds_them():
    """On made-up code: the warm-up loop as it was, a wait that counts, and one that does not."""
    load, other = ("global_load_dword", ["v0", "v[10:11]", "off"]), ("global_load_dword", ["v9", "v[10:11]", "off"])
    use, wait = ("v_mov_b32_e32", ["v4", "v0"]), lambda n: ("s_waitcnt", ["vmcnt(%d)" % n])   # noqa: E731
    end, line = ("s_endpgm", []), lambda n: [[i + 1] for i in range(n - 1)] + [[]]   # noqa: E731
    address = ("v_lshl_add_u64", ["v[10:11]", "v[0:1]", "0", "v[2:3]"])
    assert _touched_in_flight("k", [address, load, ("s_cbranch_execnz", ["0"]), wait(0), end], [[1], [2], [0, 3], [4], []])
    assert not _touched_in_flight("k", [load, other, wait(1), use, end], line(5))
    assert _touched_in_flight("k", [load, other, wait(2), use, end], line(5))
    assert _touched_in_flight("k", [load, ("s_waitcnt", ["lgkmcnt(0)"]), use, end], line(4))


def test_the_search_for_early_reads_finds_them():
    """On made-up code: straight on, with enough waiting, and around a loop."""
    mfma = ("v_mfma_f32_32x32x2_f32", ["a[0:15]", "v1", "v2", "a[0:15]"])
    read = ("v_accvgpr_read_b32", ["v17", "a15"])
    end = ("s_endpgm", [])
    line = lambda n: [[i + 1] for i in range(n - 1)] + [[]]   # noqa: E731
    assert _early_uses("k", [mfma, ("s_nop", ["7"]), read, end], line(4))
    assert not _early_uses("k", [mfma, ("s_nop", ["15"]), ("s_nop", ["1"]), read, end], line(5))
    assert _early_uses("k", [read, mfma, ("s_cbranch_scc1", ["0"]), end], [[1], [2], [0, 3], []])
