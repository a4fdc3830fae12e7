import os
"""Build-time checks on the gfx950 code objects (no GPU needed: hipcc cross-compiles, llvm-objdump / llvm-readelf read
the result).

Several kernels issue global loads from inline asm that the compiler does not track and cover them with hand-counted
`s_waitcnt vmcnt(N)` (ssdk::gload16_async for the Q fragments of the attention kernels; the C.B^T and dt loads of the
head-per-wave scan).  That is only sound while the compiler never saves or copies the destination registers between the
load and the wait — i.e. while the kernel SPILLS NOTHING: a spilled register with a load in flight is stored before its
data arrives and reloaded stale (this happened in a spilling scan kernel, since removed).
So every kernel that uses the idiom must have zero scratch; a compiler upgrade or a source edit that introduces a spill
fails here instead of producing silently wrong numbers on the GPU."""
import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

from timeviper_amd import build

ROOT = Path(__file__).resolve().parent.parent
LLVM = Path("/opt/rocm/lib/llvm/bin")
needs_tools = pytest.mark.skipif(not (LLVM / "llvm-objdump").exists() or not (LLVM / "llvm-readelf").exists(),
                                 reason="ROCm LLVM tools not found")


def kernel_metadata(src_name: str, tmp_path: Path) -> dict:
    """{mangled kernel name: {private_segment_fixed_size, vgpr_spill_count, ...}} of lib/obj/<src>.o"""
    build.ensure_built()
    obj = build.OBJ / (src_name + ".o")
    work = tmp_path / src_name
    work.mkdir()
    shutil.copy(obj, work / obj.name)                      # llvm-objdump --offloading writes next to its input
    subprocess.run([str(LLVM / "llvm-objdump"), "--offloading", obj.name], cwd=work, check=True, capture_output=True)
    dev = [p for p in work.iterdir() if "amdgcn" in p.name]
    assert len(dev) == 1, [p.name for p in work.iterdir()]
    notes = subprocess.run([str(LLVM / "llvm-readelf"), "--notes", dev[0].name], cwd=work, check=True,
                           capture_output=True, text=True).stdout
    out, cur = {}, None
    for line in notes.splitlines():
        m = re.match(r"\s*-?\s*\.(\w+):\s*(\S+)", line)
        if not m:
            continue
        key, val = m.group(1), m.group(2)
        if key == "name" and val.startswith("_Z"):
            cur = out.setdefault(val, {})
        elif cur is not None and key in ("private_segment_fixed_size", "vgpr_spill_count", "sgpr_spill_count",
                                         "vgpr_count", "agpr_count"):
            cur[key] = int(val)
    # (.name comes after the counts inside one kernel's block in some LLVM versions: collect per block instead)
    blocks = re.split(r"\n\s*- \.agpr_count:", notes)
    for b in blocks[1:]:
        name = re.search(r"\.name:\s*(_Z\S+)", b)
        if not name:
            continue
        d = out.setdefault(name.group(1), {})
        for key in ("private_segment_fixed_size", "vgpr_spill_count", "sgpr_spill_count", "vgpr_count"):
            m = re.search(r"\." + key + r":\s*(\d+)", b)
            if m:
                d[key] = int(m.group(1))
    return out


@needs_tools
def test_head_scan_fast_kernels_spill_nothing(tmp_path):
    """ssd_head_kernel<PT, 4, 2> (the kernels that run in the 9B model) carry untracked loads: zero scratch."""
    md = kernel_metadata("ssd_head.hip", tmp_path)
    fast4 = {k: v for k, v in md.items() if re.search(r"ssd_head_kernelILi\dELi4ELi2E", k)}
    assert len(fast4) >= 3, list(md)
    asm = tmp_path / "ssd_head.s"
    subprocess.run([build.HIPCC, *build.FLAGS, f"-I{build.CSRC}", "-x", "hip", "-S", "--cuda-device-only",
                    str(build.CSRC / "ssd_head.hip"), "-o", str(asm)], check=True, capture_output=True)
    text = asm.read_text()
    for k, v in fast4.items():
        # (scalar spills into vector lanes may leave a reserved, never touched stack slot behind: what counts is that no
        # instruction of the kernel reads or writes scratch memory)
        body = text[text.index(f"\n{k}:"):]
        body = body[:body.index(".amdhsa_kernel")]
        assert "scratch_" not in body and v.get("vgpr_spill_count", 0) == 0, (k, v)
    # (the variants with fewer waves per work-group may spill: they use ordinary loads)


@needs_tools
def test_head_scan_asm_kernel_spills_nothing_and_keeps_out_of_the_body_s_registers(tmp_path):
    """ssd_head_asm_kernel (head_dim 80 x 4 heads: the 9B model's scan) keeps its state in a0..a159 and the step body's
    values in v76..v255 ACROSS statements the compiler cannot see into (csrc/ssd_head_step.inc).  That holds only while
    the compiler itself never touches those registers between the statements: no scratch, no v_accvgpr_* / AGPR operand
    and no VGPR >= TV_HEAD_STEP_V0 outside ;;#ASMSTART .. ;;#ASMEND."""
    md = kernel_metadata("ssd_head.hip", tmp_path)
    k = [v for n, v in md.items() if "ssd_head_asm_kernel" in n]
    assert len(k) == 1, list(md)
    assert k[0].get("private_segment_fixed_size") == 0 and k[0].get("vgpr_spill_count", 0) == 0, k[0]
    inc = (build.CSRC / "ssd_head_step.inc").read_text()
    v0 = int(re.search(r"#define TV_HEAD_STEP_V0 (\d+)", inc).group(1))
    asm = tmp_path / "ssd_head.s"
    subprocess.run([build.HIPCC, *build.FLAGS, f"-I{build.CSRC}", "-x", "hip", "-S", "--cuda-device-only",
                    str(build.CSRC / "ssd_head.hip"), "-o", str(asm)], check=True, capture_output=True)
    text = asm.read_text()
    body = text[text.index("ssd_head_asm_kernel"):]
    body = body[body.index(": ; @"):body.index(".amdhsa_kernel")]
    inside, bad = False, []
    for line in body.splitlines():
        if "#ASMSTART" in line:
            inside = True
        elif "#ASMEND" in line:
            inside = False
        elif not inside:
            t = line.strip()
            if not t or t.startswith((";", ".")):
                continue
            regs = [int(a or c) for a, b, c in re.findall(r"\bv(\d+)\b|v\[(\d+):(\d+)\]", t)]
            if "accvgpr" in t or re.search(r"\ba\[?\d", t) or "scratch_" in t or any(r >= v0 for r in regs):
                bad.append(t)
    assert not bad, bad[:5]


def test_head_step_include_is_what_the_generator_writes():
    """csrc/ssd_head_step.inc is generated (devtools/gen_head_step.py --scalar): the committed file must be the generator's
    output, so that the schedule, the register map and the wait counts can be read (and changed) in one place."""
    import sys
    out = subprocess.run([sys.executable, str(build.ROOT / "devtools" / "gen_head_step.py"), "--scalar"], check=True,
                         capture_output=True, text=True).stdout
    assert out == (build.CSRC / "ssd_head_step.inc").read_text()


@needs_tools
def test_attention_kernels_with_untracked_q_loads_spill_nothing(tmp_path):
    """flash_fwd_kernel / flash_fwd_stream_kernel load their Q fragments with ssdk::gload16_async."""
    for src in ("attention.hip", "attention_fp8.hip"):
        text = (build.CSRC / src).read_text()
        if "gload16_async" not in text:
            continue
        md = kernel_metadata(src, tmp_path)
        kernels = {k: v for k, v in md.items() if "flash_fwd" in k}
        assert kernels, (src, list(md))
        for k, v in kernels.items():
            assert v.get("private_segment_fixed_size") == 0 and v.get("vgpr_spill_count", 0) == 0, (src, k, v)


@needs_tools
def test_gemm_kernels_spill_nothing(tmp_path):
    """Both GEMM kernels keep five half-tiles of LDS-DMA copies in flight behind hand-counted waits and, at two waves per
    SIMD, live within 256 registers: a spill would put scratch loads — which the compiler waits for with vmcnt(0) — into
    the copy queue and drain the pipeline every K-tile.  (Scalar spills into vector lanes are allowed: no memory.)"""
    for src, pat, n in (("gemm.hip", "gemm_bf16_kernel", 5), ("gemm_persist.hip", "gemm_persist_kernel", 2),
                        ("gemm_drip.hip", "gemm_drip_kernel", 3)):
        md = kernel_metadata(src, tmp_path)
        kernels = {k: v for k, v in md.items() if pat in k}
        assert len(kernels) == n, (src, list(md))
        for k, v in kernels.items():
            assert v.get("private_segment_fixed_size") == 0 and v.get("vgpr_spill_count", 0) == 0, (src, k, v)


def test_gemm_drip_register_statements_are_current():
    """csrc/gemm_drip_regs.inc (the statements of the 256 x 192 GEMM that name accumulator registers) is what
    devtools/gen_gemm_drip_regs.py emits."""
    r = subprocess.run([sys.executable, str(ROOT / "timeviper_amd" / "devtools" / "gen_gemm_drip_regs.py"), "--check"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


@needs_tools
def test_gemm_drip_accumulator_registers_are_left_alone(tmp_path):
    """gemm_drip.hip keeps its accumulators (a[0:95]) and the parked half of the finished tile (a[96:119]) in registers the
    compiler does not allocate: outside the hand-written statements the compiled kernel must not touch an accumulator
    register (it is built with -amdgpu-spill-vgpr-to-agpr=0 for that reason), and it must use no scratch."""
    src = ROOT / "timeviper_amd" / "csrc" / "gemm_drip.hip"
    out = tmp_path / "gemm_drip.s"
    flags = [f for f in build.FLAGS if not f.startswith("-fPIC")] + build.FILE_FLAGS["gemm_drip.hip"]
    r = subprocess.run([build.HIPCC, *flags, "-x", "hip", "-S", "--cuda-device-only", str(src), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    inasm, bad = False, []
    for ln in out.read_text().splitlines():
        if "#ASMSTART" in ln:
            inasm = True
        elif "#ASMEND" in ln:
            inasm = False
        elif not inasm and not ln.lstrip().startswith((";", ".")) and re.search(r"[\s,\[]a\[?\d", ln):
            bad.append(ln.strip())
        if "scratch_" in ln:
            bad.append(ln.strip())
    assert not bad, bad[:10]

@needs_tools
def test_vit_attention_asm_kernel_keeps_out_of_the_body_s_registers(tmp_path):
    """flash_fwd_vit_kernel (csrc/attention_vit.hpp) keeps P, the running maxima (v[TV_FAV_V0 ..]) and O / S / Q (a0 .. a231)
    in named registers ACROSS the statements of a query block: between the block's first statement (TV_FAV_BEGIN_ASM) and
    its last (TV_FAV_EPI_ASM) the compiler must use no vector register >= TV_FAV_V0 and no accumulation register below
    232, and the kernel must have no scratch."""
    md = kernel_metadata("attention.hip", tmp_path)
    k = [v for n, v in md.items() if "flash_fwd_vit_kernel" in n]
    assert len(k) == 1, list(md)
    assert k[0].get("private_segment_fixed_size") == 0 and k[0].get("vgpr_spill_count", 0) == 0, k[0]
    inc = (build.CSRC / "attention_vit_tile.inc").read_text()
    v0 = int(re.search(r"#define TV_FAV_V0 (\d+)", inc).group(1))
    asm = tmp_path / "attention.s"
    subprocess.run([build.HIPCC, *build.FLAGS, f"-I{build.CSRC}", "-x", "hip", "-S", "--cuda-device-only",
                    str(build.CSRC / "attention.hip"), "-o", str(asm)], check=True, capture_output=True)
    text = asm.read_text()
    body = text[text.index("flash_fwd_vit_kernel"):]
    body = body[body.index(": ; @"):body.index(".amdhsa_kernel")]
    inside, in_block, cur, bad = False, False, [], []
    for line in body.splitlines():
        if "#ASMSTART" in line:
            inside, cur = True, []
        elif "#ASMEND" in line:
            inside = False
            big = len(cur) > 40
            mfmas = sum("v_mfma" in c for c in cur)
            if big and mfmas == 0 and any("v_accvgpr_write_b32 a0, 0" in c for c in cur):
                in_block = True                       # TV_FAV_BEGIN_ASM
            elif big and mfmas == 36 and not any("v_exp_f32" in c for c in cur):
                in_block = False                      # TV_FAV_EPI_ASM
        elif inside:
            cur.append(line)
        elif in_block:
            t = line.strip()
            if not t or t.startswith((";", ".")):
                continue
            regs = [int(a or c) for a, b, c in re.findall(r"\bv(\d+)\b|v\[(\d+):(\d+)\]", t)]
            aregs = [int(a or c) for a, b, c in re.findall(r"\ba(\d+)\b|a\[(\d+):(\d+)\]", t)]
            if "scratch_" in t or any(r >= v0 for r in regs) or any(r < 232 for r in aregs):
                bad.append(t)
    assert not bad, bad[:5]


def test_vit_attention_tile_include_is_what_the_generator_writes():
    """csrc/attention_vit_tile.inc is generated (devtools/gen_fa_vit.py)."""
    import sys
    out = subprocess.run([sys.executable, str(build.ROOT / "devtools" / "gen_fa_vit.py")], check=True, capture_output=True,
                         text=True, env={k: v for k, v in os.environ.items() if k != "TV_FAV_ABLATE"}).stdout
    assert out == (build.CSRC / "attention_vit_tile.inc").read_text()


# ---- wait states that the hardware does not keep by itself, counted in the built code.  The compiler keeps them for its own instructions; it does not look into
# the inline statements (copies into LDS, stores), so a v_readfirstlane that it puts right in front of one is seen only here.
def _registers(text: str, kind: str) -> set:
    out = set()
    for m in re.finditer(rf"(?<![\w\[:])([{kind}])(\d+)\b|\b([{kind}])\[(\d+):(\d+)\]|\b(vcc|m0)\b", text):
        if m.group(1):
            out.add(m.group(1) + m.group(2))
        elif m.group(3):
            out.update(f"{m.group(3)}{i}" for i in range(int(m.group(4)), int(m.group(5)) + 1))
        elif "s" in kind:
            out.add(m.group(6))
    return out


class _Instruction:
    __slots__ = ("op", "ops", "at", "next", "states", "of")

    def __init__(self, op, args, at, of=None):
        self.op, self.at, self.next, self.of = op, at, [], of
        self.ops = [o.strip() for o in re.split(r",(?![^\[]*\])", args)] if args else []
        self.states = int(self.ops[0], 0) + 1 if op == "s_nop" else 1


def _device_code(src_name: str, work: Path) -> list:
    """The instructions of lib/obj/<src>.o in order, each with what can follow it"""
    work.mkdir()
    obj = build.OBJ / (src_name + ".o")
    shutil.copy(obj, work / obj.name)
    subprocess.run([str(LLVM / "llvm-objdump"), "--offloading", obj.name], cwd=work, check=True, capture_output=True)
    out, symbols, jumps, of = [], {}, [], None
    for dev in (p for p in work.iterdir() if "amdgcn" in p.name):
        for line in subprocess.run([str(LLVM / "llvm-objdump"), "-d", dev.name], cwd=work, check=True, capture_output=True, text=True).stdout.splitlines():
            if m := re.match(r"([0-9a-f]+) <(.+)>:", line):
                of = m.group(2)
                symbols[of] = int(m.group(1), 16)
            elif m := re.match(r"\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):\s*(.*)$", line):
                out.append(_Instruction(m.group(1), m.group(2), int(m.group(3), 16), of))
                t = re.search(r"<([^>+]+)(?:\+0x([0-9a-f]+))?>", m.group(4))
                if t and m.group(1).startswith(("s_branch", "s_cbranch")):
                    jumps.append((len(out) - 1, t.group(1), int(t.group(2) or "0", 16)))
    where = {i.at: i for i in out}
    for a, b in zip(out, out[1:]):
        if a.op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
            a.next.append(b)
    for n, name, offset in jumps:
        out[n].next.append(where[symbols[name] + offset])
    return out


def _too_near(first: _Instruction, live: set, need: int, reads, writes) -> list:
    """The instructions that read one of `live`, written by `first`, with fewer than `need` wait states between, on any path"""
    found, seen, todo = [], {}, [(n, 0, frozenset(live)) for n in first.next]
    while todo:
        i, passed, regs = todo.pop()
        if passed >= need or not regs or seen.get((i.at, regs), need) <= passed:
            continue
        seen[i.at, regs] = passed
        if reads(i) & regs:
            found.append((passed, i))
        todo += [(n, passed + i.states, regs - writes(i)) for n in i.next]
    return found


@pytest.fixture(scope="module")
def device_code(tmp_path_factory):
    """{source: its instructions}"""
    build.ensure_built()
    work = tmp_path_factory.mktemp("device")
    return {src.name: _device_code(src.name, work / src.name) for src in build._sources()}


_MEMORY = ("global_", "buffer_", "flat_", "scratch_")


def _scalar_results(i: _Instruction) -> set:
    """Scalar registers that a vector instruction writes"""
    if i.op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
        return _registers(i.ops[0], "s")
    if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[ui]64", i.op):
        return _registers(i.ops[1], "s")
    return set()


def _scalar_writes(i: _Instruction) -> set:
    if i.op.startswith("s_") and i.ops and not i.op.startswith(("s_cmp", "s_bitcmp", "s_waitcnt", "s_nop", "s_cbranch", "s_branch", "s_set")):
        return _registers(i.ops[0], "s")
    return _scalar_results(i)


@needs_tools
def test_loads_keep_five_wait_states_behind_a_vector_write_of_their_scalar_address(device_code):
    """A vector-memory instruction that reads a scalar register (address, M0 aside) which v_readfirstlane, v_readlane or a compare has written reads the old value
    within five wait states."""
    bad = []
    for src, code in device_code.items():
        for i in code:
            if live := _scalar_results(i):
                for passed, j in _too_near(i, live, 5, lambda k: _registers(" ".join(k.ops), "s") if k.op.startswith(_MEMORY) else set(), _scalar_writes):
                    bad.append((src, passed, i.op, i.ops, j.op, j.ops))
    assert not bad, (len(bad), bad[:4])


def _vector_writes(i: _Instruction) -> set:
    return _registers(i.ops[0], "va") if i.op.startswith("v_") and i.ops else set()


@needs_tools
def test_wide_stores_keep_their_data_for_two_wait_states(device_code):
    """A store of more than 8 bytes still reads its data in the two wait states behind it: no vector instruction may write those registers there."""
    bad = []
    for src, code in device_code.items():
        for i in code:
            if re.match(r"(global|flat|buffer)_store_dwordx[34]$", i.op):
                data = i.ops[0 if i.op.startswith("buffer") else 1]
                for passed, j in _too_near(i, _registers(data, "va"), 2, _vector_writes, lambda k: set()):
                    bad.append((src, passed, i.op, i.ops, j.op, j.ops))
    assert not bad, (len(bad), bad[:4])


def test_the_count_of_wait_states_sees_what_is_too_near():
    def code(*lines):
        out = [_Instruction(*(ln.split(" ", 1) + [""])[:2], n) for n, ln in enumerate(lines)]
        for a, b in zip(out, out[1:]):
            a.next.append(b)
        return out

    def near(*lines):
        c = code(*lines)
        return [p for p, _ in _too_near(c[0], _scalar_results(c[0]), 5, lambda k: _registers(" ".join(k.ops), "s") if k.op.startswith(_MEMORY) else set(), _scalar_writes)]
    head = ("s_mov_b32 s9, m0", "s_mov_b32 m0, s8")
    assert near("v_readfirstlane_b32 s5, v1", *head, "s_nop 0", "global_load_lds_dwordx4 v0, s[4:5]") == [3]
    assert near("v_readfirstlane_b32 s5, v1", *head, "s_nop 2", "global_load_lds_dwordx4 v0, s[4:5]") == []
    assert near("v_readlane_b32 s4, v1, 3", "s_add_u32 s4, s4, s6", "global_load_dwordx4 v[0:3], v0, s[4:5] offset:16") == []
    assert near("v_cmp_gt_u32_e64 s[4:5], v1, v2", "global_store_dwordx4 v0, v[4:7], s[4:5]") == [0]


@needs_tools
def test_an_attention_step_copies_its_pieces_once(device_code):
    """flash_fwd_kernel with two tiles a step: as many copies whatever the head dim, whose MFMAs they stand between"""
    copies = {}
    for i in device_code["attention.hip"]:
        if m := re.match(r"_ZN12_GLOBAL__N_116flash_fwd_kernelI(\w+)Li\dELi\dELi8ELi2ELb(\d)ELi(\d)E", i.of or ""):
            copies.setdefault(m.groups(), {}).setdefault(i.of, 0)
            copies[m.groups()][i.of] += "_lds_" in i.op
    assert len(copies) == 6 and all(len(k) >= 3 and len(set(k.values())) == 1 for k in copies.values()), copies
