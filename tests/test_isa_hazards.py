"""Static check of the generated gfx950 code of the MFMA kernels (no GPU needed: hipcc cross-compiles).

The kernels issue their direct-to-LDS loads from inline assembly with the base address in scalar registers.  On
gfx9-family hardware a vector memory instruction must not read a scalar register within five wait states of a
vector instruction (v_readfirstlane, v_readlane) writing it; the compiler keeps that distance for its own instructions but does
not look into assembly blocks, and a load that reads a stale base faults the GPU.  The test compiles every
source of the MFMA kernels to assembly and looks at the six instructions in front of every load of an assembly block."""
import os
import re
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

from scattermoe_amd import _build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
VMEM = re.compile(r"\b(global_load|buffer_load|global_store|buffer_store)\w*\b")
SCALAR = re.compile(r"\bs(?:(\d+)\b|\[(\d+):(\d+)\])")      # base, descriptor, scalar offset
VALU_TO_SGPR = re.compile(r"v_\w+ s(?:(\d+)|\[(\d+):(\d+)\])")      # a vector instruction whose destination is scalar


def _hazards(text):
    lines = text.split("\n")
    found, loads, inside = [], 0, False
    for i, line in enumerate(lines):
        if "ASMSTART" in line:
            inside = True
            continue
        if "ASMEND" in line:
            inside = False
            continue
        if not (inside and VMEM.search(line)):
            continue
        regs = set()
        for m in SCALAR.finditer(line):
            regs |= set(range(int(m[1] or m[2]), int(m[1] or m[3]) + 1))
        if not regs:
            continue
        loads += 1
        k, states = i - 1, 0
        while k >= 0 and states < 6:
            t = lines[k].strip()
            k -= 1
            if not t or t[0] in ";." or t.endswith(":"):
                continue
            nop = re.match(r"s_nop (\d+)", t)
            states += int(nop.group(1)) + 1 if nop else 1
            w = VALU_TO_SGPR.match(t)
            if w and states <= 5 and regs & set(range(int(w[1] or w[2]), int(w[1] or w[3]) + 1)):
                found.append((i + 1, t, line.strip()))
                break
    return loads, found


def test_scanner_sees_a_hazard_and_its_fix():
    bad = "\tv_readfirstlane_b32 s2, v20\n\t;;#ASMSTART\n\tglobal_load_dword v1, v2, s[2:3]\n\t;;#ASMEND\n"
    good = "\tv_readfirstlane_b32 s2, v20\n\t;;#ASMSTART\n\ts_nop 4\n\tglobal_load_dword v1, v2, s[2:3]\n\t;;#ASMEND\n"
    assert _hazards(bad)[1] and not _hazards(good)[1]
    for writer in ("v_readlane_b32 s3, v20, s9", "v_cmp_lt_u32_e64 s[2:3], v1, v2", "v_readlane_b32 s2, v20, 63"):
        assert _hazards(bad.replace("v_readfirstlane_b32 s2, v20", writer))[1], writer
    assert not _hazards(bad.replace("v_readfirstlane_b32 s2, v20", "v_readlane_b32 s4, v20, s2"))[1]
    for load in ("buffer_load_dwordx4 v1, s[4:7], s2 offen lds", "buffer_load_dwordx4 v1, s[0:3], s6 offen lds"):
        assert _hazards(bad.replace("global_load_dword v1, v2, s[2:3]", load))[1], load
        assert not _hazards(good.replace("global_load_dword v1, v2, s[2:3]", load))[1], load
    assert not _hazards(bad.replace("global_load_dword v1, v2, s[2:3]", "buffer_load_dwordx4 v1, s[4:7], s3 offen lds"))[1]


def _sources():
    """Every compiled source that instantiates the MFMA kernels."""
    names = [n for n in _build.SOURCES if "gemm_mfma.hpp" in open(os.path.join(_build.CSRC, n)).read()]
    assert len(names) >= 3
    return names


VECTOR = re.compile(r"\b([av])(?:(\d+)\b|\[(\d+):(\d+)\])")


def _vector_registers(text):
    return {(m[1], k) for m in VECTOR.finditer(text) for k in range(int(m[2] or m[3]), int(m[2] or m[4]) + 1)}


def _product_hazards(text):
    """Products issued from assembly blocks, which the compiler's hazard recogniser does not look into: a vector instruction
    must not write one of their operands within the two wait states before them, and nothing but a product may touch their
    result within the 19 states that the longest of them takes to write it (followed in program order, as the code falls
    through)."""
    code, inside = [], False
    for n, line in enumerate(text.split("\n")):
        t = line.strip()
        if "ASMSTART" in t or "ASMEND" in t:
            inside = "ASMSTART" in t
        elif t and t[0] not in ".;" and not t.split(";")[0].strip().endswith(":"):
            code.append((n + 1, t.split(";")[0].strip(), inside))
    states = lambda t: int(t.split()[1]) + 1 if t.startswith("s_nop") else 1
    products, found = 0, []
    for i, (n, t, in_asm) in enumerate(code):
        if not (in_asm and t.startswith("v_mfma")):
            continue
        products += 1
        operands = t.split(None, 1)[1].split(",")
        result, sources = _vector_registers(operands[0]), _vector_registers(",".join(operands[1:]))
        k, passed = i - 1, 0
        while k >= 0 and passed < 2:
            u = code[k][1]
            if u.startswith("v_") and not u.startswith("v_mfma") and _vector_registers(u.split(",")[0]) & sources:
                found.append((n, t, code[k]))
            passed, k = passed + states(u), k - 1
        k, passed = i + 1, 0
        while k < len(code) and passed < 19 and not code[k][1].startswith(("s_branch", "s_endpgm", "s_setpc")):
            u = code[k][1]
            if not u.startswith("v_mfma") and _vector_registers(u) & result:
                found.append((n, t, code[k]))
            passed, k = passed + states(u), k + 1
    return products, found


def test_scanner_sees_an_early_access_of_a_product():
    product = "\t;;#ASMSTART\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[4:7], a[0:3]\n\t;;#ASMEND\n"
    for bad in ("\tv_mov_b32_e32 v5, v1\n" + product, "\tv_accvgpr_write_b32 a3, 0\n\ts_nop 0\n" + product,
                product + "\tv_accvgpr_read_b32 v1, a2\n", product + "\ts_nop 15\n\tscratch_store_dword off, a3, off\n",
                product + ".LBB0_1:\n\tv_mov_b32_e32 v9, v1\n\tv_accvgpr_read_b32 v1, a0\n"):
        assert _product_hazards(bad)[1], bad
    for good in ("\tv_mov_b32_e32 v5, v1\n\ts_nop 1\n" + product, product + product, "\tv_mov_b32_e32 v3, v5\n" + product,
                 product + "\ts_nop 15\n\ts_nop 3\n\tv_accvgpr_read_b32 v1, a2\n", product + "\tds_read_b128 v[8:11], v1\n"):
        assert _product_hazards(good) == (good.count("v_mfma"), []), good


needs_hipcc = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"),
                                 reason="needs hipcc")


@pytest.fixture(scope="module")
def assembly():
    """File name -> generated assembly of the sources that instantiate the MFMA kernels."""
    names = _sources()
    with tempfile.TemporaryDirectory() as tmp:
        def compile_(name):
            out = os.path.join(tmp, name + ".s")
            cmd = [_build._hipcc()] + _build.HIPCC_FLAGS + ["-S", "--cuda-device-only", "-o", out,
                                                           os.path.join(_build.CSRC, name)]
            subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
            return open(out).read()
        with ThreadPoolExecutor(max_workers=len(names)) as pool:      # side by side
            return dict(zip(names, pool.map(compile_, names)))


@needs_hipcc
def test_no_inline_assembly_load_reads_a_freshly_written_scalar_base(assembly):
    for name, text in assembly.items():
        loads, found = _hazards(text)
        assert loads > 100, "%s: no inline-assembly loads found: the scan is looking at the wrong text" % name
        assert not found, (name, found[:5])


@needs_hipcc
def test_products_of_assembly_blocks_keep_their_distance(assembly):
    seen = 0
    for name, text in assembly.items():
        products, found = _product_hazards(text)
        seen += products
        assert not found, (name, found[:5])
    assert seen > 1000, "no inline-assembly products found: the scan is looking at the wrong text"


def _scratch_of_kernels(text):
    """(name, bytes of scratch memory per lane) of every kernel of an assembly listing, from its metadata."""
    out = []
    for block in text.split("\n  - .agpr_count:")[1:]:
        name, size = (re.search(r"\.%s:\s+(\S+)" % k, block).group(1) for k in ("name", "private_segment_fixed_size"))
        out.append((name, int(size)))
    return out


def _tile(name):
    """The Tile<...> arguments in a kernel's mangled name: (BM, BN, WM, WN, NS, RS, ...)."""
    m = re.search(r"4TileI((?:L[ib]\d+E)+)E", name)
    return tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1))) if m else ()


@needs_hipcc
def test_kernels_fit_their_registers(assembly):
    """What does not fit goes to scratch memory, for every thread of every tile.  Five registers at the most (gathered
    rows in 128 x 128 tiles, four workgroups per CU), three in the one-wave-per-SIMD form of scatter2scatter, which has
    256 accumulators and two register sets of operands, and none of those in the path of a full tile."""
    seen = 0
    for name, text in assembly.items():
        for kernel, scratch in _scratch_of_kernels(text):
            one_wave = "s2s_mfma_kernel" in kernel and _tile(kernel)[:6] == (256, 256, 2, 2, 2, 1)
            seen += one_wave
            assert scratch <= (12 if one_wave else 20), (name, kernel, scratch)
    assert seen == 4


JUMP = re.compile(r"s_c?branch\w*\s+(\S+)")


def _product_hazards_on_all_paths(text):
    """As `_product_hazards`, along every path that the code can take: both ways of a branch, a loop's back edge among them, and every
    jump that leads to a product."""
    code, labels, inside = [], {}, False
    for n, line in enumerate(text.split("\n")):
        t = line.split(";")[0].strip()
        if "ASMSTART" in line or "ASMEND" in line:
            inside = "ASMSTART" in line
        elif t.endswith(":"):
            labels[t[:-1]] = len(code)
        elif t and t[0] != ".":
            code.append((n + 1, t, inside))
    ends = lambda t: t.startswith(("s_branch", "s_endpgm", "s_setpc"))
    jump = lambda t: JUMP.match(t) and labels[JUMP.match(t)[1]]
    after, before = [], [[] for _ in code]
    for i, (_, t, _) in enumerate(code):
        to = [k for k in (None if ends(t) else i + 1, jump(t)) if k is not None and k < len(code)]
        after.append(to)
        for k in to:
            before[k].append(i)
    states = lambda t: int(t.split()[1]) + 1 if t.startswith("s_nop") else 1

    def reached(start, edges, limit):
        """Instructions that fewer than `limit` wait states lie between."""
        least, todo = {}, [(k, 0) for k in edges[start]]
        while todo:
            k, passed = todo.pop()
            if passed < limit and passed < least.get(k, limit):
                least[k] = passed
                todo += [(j, passed + states(code[k][1])) for j in edges[k]]
        return least

    products, found = 0, []
    for i, (n, t, in_asm) in enumerate(code):
        if not (in_asm and t.startswith("v_mfma")):
            continue
        products += 1
        operands = t.split(None, 1)[1].split(",")
        result, sources = _vector_registers(operands[0]), _vector_registers(",".join(operands[1:]))
        found += [(n, t, code[k]) for k in reached(i, before, 2) if code[k][1].startswith("v_") and
                  not code[k][1].startswith("v_mfma") and _vector_registers(code[k][1].split(",")[0]) & sources]
        found += [(n, t, code[k]) for k in reached(i, after, 19)
                  if not code[k][1].startswith("v_mfma") and _vector_registers(code[k][1]) & result]
    return products, found


def test_scanner_follows_branches():
    product = "\t;;#ASMSTART\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[4:7], a[0:3]\n\t;;#ASMEND\n"
    loop = ".LBB0_1:                                ; loop\n%s" + product + "%s\ts_cbranch_scc1 .LBB0_1\n%s\ts_endpgm\n"
    skip = product + "\ts_cbranch_scc0 .LBB0_2\n\ts_nop 15\n\ts_nop 3\n%s.LBB0_2:\n%s\ts_endpgm\n"
    enter = "\tv_mov_b32_e32 v5, v1\n\ts_branch .LBB0_3\n\ts_endpgm\n.LBB0_3:\n%s" + product
    read, wait, write = "\tv_accvgpr_read_b32 v1, a2\n", "\ts_nop 15\n\ts_nop 3\n", "\tv_mov_b32_e32 v9, v1\n"
    for bad in (loop % (read, "", wait + read), loop % ("", write, ""), loop % ("", "", read), skip % ("", read), enter % ""):
        assert _product_hazards_on_all_paths(bad)[1], bad
    # (the first two are beyond a scan of the code as it falls through)
    assert not _product_hazards(loop % (read, "", wait + read))[1] and not _product_hazards(loop % ("", write, ""))[1]
    for good in (loop % (wait + read, "", wait + read), loop % ("", write + "\ts_nop 1\n", ""), skip % (read, wait + read),
                 enter % "\ts_nop 1\n", skip % (read, "")):
        assert _product_hazards_on_all_paths(good) == (1, []), good


@needs_hipcc
def test_products_of_assembly_blocks_keep_their_distance_on_all_paths(assembly):
    for name, text in assembly.items():
        products, found = _product_hazards_on_all_paths(text)
        assert products == _product_hazards(text)[0]
        assert not found, (name, found[:5])


@needs_hipcc
def test_one_wave_per_simd_kernels_need_no_scratch_memory(assembly):
    """Products in tiles of 256 and of 192 columns, and weight gradients: 256 (192) accumulators, two register sets of operands and
    nothing in scratch memory."""
    seen = {}
    for name, text in assembly.items():
        for kernel, scratch in _scratch_of_kernels(text):
            tile = _tile(kernel)[:6]
            if tile[2:] == (2, 2, 2, 1):
                which = ("xty" if "xty_mfma_kernel" in kernel else "s2s", tile[1])
                seen[which] = seen.get(which, 0) + 1
                assert scratch == 0, (name, kernel, scratch)
    assert seen == {("s2s", 256): 4, ("s2s", 192): 4, ("xty", 256): 2}, seen
