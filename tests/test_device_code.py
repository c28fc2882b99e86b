"""Checks on the device code that hipcc makes of the panel-ring GEMM.

Its MFMAs are inline asm, so the compiler does not insert the wait states
that a read of their result needs; whether every read keeps them is a property of
the generated code, looked at here (no GPU needed).
"""

import re
import shlex
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tiktok-techjam-2026_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
# wait states between a 4-pass MFMA (16x16x32, 2-byte) and another
# instruction's use of its result on gfx950
RESULT_STATES = 8


def _panel_asm(tmp_path, elem):
    """Assembly of every plan's panel kernel (FM x FN) and epilogue, with the library's own flags."""
    src = tmp_path / f"panel_{elem}.hip"
    inst = "\n".join(
        f"template __global__ void gemm_panel_kernel<{elem}, {fm}, {fn}, {epi}>(const {elem}*, int64_t, const {elem}*, "
        f"int64_t, const {elem}*, void*, int64_t, int, int, int, ResSrc);"
        for fm, fn in ((4, 4), (3, 2), (2, 2)) for epi in (0, 1, 2, 4))
    src.write_text(f'#include "{CSRC / "gemm_kernels.h"}"\nnamespace tjk {{\n{inst}\n}}\n')
    made = subprocess.run(["make", "-n", "-B", "-C", str(CSRC), "../../_build/tjk/gemm_bf16.o"], check=True,
                          capture_output=True, text=True).stdout
    line = next(l for l in made.splitlines() if " -c " in l)
    flags = shlex.split(line.split(" -c ")[0])[1:]
    out = tmp_path / f"panel_{elem}.s"
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    return out.read_text()


def _kernels(asm):
    for m in re.finditer(r"^(_ZN3tjk17gemm_panel_kernel\S+):", asm, re.M):
        body = asm[m.end():asm.index(".Lfunc_end", m.end())]
        lines = [l.split(";")[0].strip() for l in body.splitlines()]
        yield m.group(1), [l for l in lines if l and (not l.startswith(".") or l.endswith(":"))]


def _agprs(text):
    regs = set()
    for lo, hi, one in re.findall(r"\ba(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        regs |= set(range(int(lo), int(hi) + 1)) if lo else {int(one)}
    return regs


def _early_uses(code):
    """(MFMA, instruction) pairs where the instruction touches the MFMA's result
    within RESULT_STATES, along every path; an instruction counts as one state,
    s_nop N as N + 1, time spent at a barrier as none."""
    label = {l[:-1]: i for i, l in enumerate(code) if l.endswith(":")}
    bad = []
    for start, mfma in enumerate(code):
        if not mfma.startswith("v_mfma"):
            continue
        dest = _agprs(mfma.split(",")[0])
        paths, seen = [(start + 1, RESULT_STATES)], set()
        while paths:
            i, left = paths.pop()
            while left > 0 and i < len(code) and (i, left) not in seen:
                seen.add((i, left))
                l = code[i]
                if l.endswith(":"):
                    i += 1
                    continue
                if not l.startswith("v_mfma") and _agprs(l) & dest:
                    bad.append((mfma, l))
                    break
                left -= int(l.split()[1]) + 1 if l.startswith("s_nop") else 1
                if l.startswith("s_endpgm"):
                    break
                if l.startswith(("s_branch", "s_cbranch")):
                    paths.append((label[l.split()[1]], left))
                    if l.startswith("s_branch"):
                        break
                i += 1
    return bad


def test_early_use_is_found():
    mfma = "v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[4:7]"
    read = "v_accvgpr_read_b32 v1, a6"
    assert _early_uses([mfma, "s_nop 5", "s_barrier", read])
    assert not _early_uses([mfma, "s_nop 6", "s_barrier", read])
    assert not _early_uses([mfma, "v_accvgpr_read_b32 v1, a8"])
    assert _early_uses(["L:", read, "s_nop 7", mfma, "s_cbranch_scc1 L"])


@pytest.mark.skipif(not Path(HIPCC).exists() or shutil.which("make") is None, reason="needs hipcc and make")
@pytest.mark.parametrize("elem", ["bf16", "f16"])
def test_panel_gemm_reads_results_after_their_wait(tmp_path, elem):
    """Every instance: no read of an accumulator before the MFMA that wrote it
    is done, and no scratch (a spilled accumulator is such a read)."""
    asm = _panel_asm(tmp_path, elem)
    kernels = dict(_kernels(asm))
    assert len(kernels) == 12
    for name, code in kernels.items():
        assert sum(l.startswith("v_mfma") for l in code) >= 8, name
        assert not _early_uses(code), (name, _early_uses(code)[:3])
        assert not any(l.startswith("scratch_") for l in code), name


OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
LIB = CSRC.parent / "tjkernels" / "libtjk.so"


def _library_kernels(tmp_path, lib, what):
    """(name, instructions) of the kernels named `what` in a built library."""
    copy = tmp_path / "lib.so"
    shutil.copy(lib, copy)
    subprocess.run([OBJDUMP, "--offloading", str(copy)], check=True, capture_output=True, cwd=tmp_path)
    for part in sorted(tmp_path.glob("lib.so.*gfx950*")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(part)], check=True,
                              capture_output=True, text=True).stdout
        for m in re.finditer(r"^<(\S*" + what + r"\S*)>:\n((?:\t.*\n)+)", text, re.M):
            yield m.group(1), [l.split("//")[0].strip() for l in m.group(2).splitlines()]


@pytest.fixture(scope="module")
def attention_rings(tmp_path_factory):
    """{MASK: {name: instructions up to the first copy into LDS}} of the built
    attention kernels whose K / V ring is filled by copies (4 or 8 waves)."""
    if not Path(OBJDUMP).exists() or not LIB.exists():
        pytest.skip("needs llvm-objdump and the built library")
    rings = {}
    for name, code in _library_kernels(tmp_path_factory.mktemp("lib"), LIB, "flash_pipe_kernelI"):
        mask = int(re.search(r"ELi(\d)ELi[48]EEE", name).group(1))
        first = [i for i, l in enumerate(code) if l.startswith("buffer_load") and l.endswith("lds")]
        if first:
            rings.setdefault(mask, {})[name] = code[:first[0]]
    return rings


def test_unmasked_attention_copies_before_it_waits(attention_rings):
    """The K / V copies of a workgroup's first tiles go out before anything
    waits for a load (of Q: a memory round trip more per workgroup).  Masks 0
    and 5: kMaskNone, kMaskNoneFull."""
    assert len(attention_rings[0]) >= 8 and len(attention_rings[5]) >= 8
    # a whole head_dim of 32 takes the tiles through registers (kMaskNoneRegs)
    assert not any("Li64ELi32E" in name for name in attention_rings[5])
    for name, code in {**attention_rings[0], **attention_rings[5]}.items():
        assert not any("vmcnt" in l for l in code), name


def test_listed_attention_reads_eight_mask_blocks_at_a_time(attention_rings):
    """kMaskList (1): eight mask reads go out before the first is waited for."""
    assert len(attention_rings[1]) == 8
    for name, code in attention_rings[1].items():
        reads = [i for i, l in enumerate(code) if l.startswith("global_load_ubyte")]
        assert len(reads) == 8 and not any("vmcnt" in l for l in code[reads[0]:reads[7]]), name
