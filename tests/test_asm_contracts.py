"""Contracts of hand-written assembly that the compiler cannot check, verified
on the gfx950 assembly of this repository's own sources (no GPU needed).

load_lds16 and load_lds4 (iron_common.hpp) write M0 behind the compiler's back:
in every kernel that uses them, each M0 write must be theirs (followed by one
wait state, s_nop 0, then the buffer_load ... lds), so the compiler never keeps a
value of its own in M0 there, and no LDS-DMA load directly follows the M0 write
it reads (GFX9 needs one wait state between the two).

The compiler does not count those loads, so a vmcnt wait it inserts for a load
of its own also waits for every stage in flight: after a kernel's first LDS-DMA
load, every vmcnt wait must be one of its own, in the prefill attention right
before its barriers. Spills would bring such loads, so there are none.
"""

import functools
import re
import subprocess

import pytest

from iron_amd import _build

KERNELS = {
    "gemm.hip": ["gemm_nt_kernel", "gemm_i4_kernel", "gemm_skinny_kernel"],
    "attention.hip": ["attention_prefill_kernel", "attention_prefill_split_kernel"],
}


@functools.lru_cache(maxsize=None)
def device_asm(src_name):
    try:
        hipcc = _build._hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    src = _build.CSRC / src_name
    cmd = [hipcc, *_build.HIP_FLAGS, *_build.FILE_FLAGS.get(src_name, []), "--cuda-device-only", "-S", str(src),
           "-o", "-"]
    out = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    return out.stdout


def functions(asm):
    """name -> list of instruction lines of each function in the assembly (a
    function runs from its label to its .Lfunc_end label: it may hold several
    s_endpgm, one per exit)."""
    funcs, name, body = {}, None, []
    for line in asm.splitlines():
        m = re.match(r"^(_Z\S+):", line)
        if m:
            name, body = m.group(1), []
            funcs[name] = body
            continue
        if line.startswith(".Lfunc_end"):
            name = None
            continue
        if name is not None:
            s = line.split(";")[0].strip()
            if s and not s.startswith("."):
                body.append(s)
    return funcs


@pytest.mark.parametrize("src_name", sorted(KERNELS))
def test_m0_written_only_by_load_lds16(src_name):
    funcs = functions(device_asm(src_name))
    checked = set()
    for fname, body in funcs.items():
        kernel = next((k for k in KERNELS[src_name] if k in fname), None)
        if kernel is None:
            assert not any(re.match(r"buffer_load_\S+ .*\blds$", ins) for ins in body), fname  # it belongs in KERNELS
            continue
        checked.add(kernel)
        loads = 0
        for i, ins in enumerate(body):
            if re.search(r"\bm0\b", ins):
                assert ins.startswith("s_mov_b32 m0,"), (fname, i, ins)
                nop = body[i + 1] if i + 1 < len(body) else ""
                nxt = body[i + 2] if i + 2 < len(body) else ""
                assert nop == "s_nop 0", (fname, i, ins, nop)
                assert re.match(r"buffer_load_dword(x4)? .*\blds$", nxt), (fname, i, ins, nxt)
                loads += 1
        assert loads > 0, fname
        assert not any(ins.startswith("global_load_lds") for ins in body), fname
    assert checked == set(KERNELS[src_name])


def _own_waits(asm, name):
    """For each function of the assembly whose name holds ``name``, after its first
    LDS-DMA load: the vmcnt waits that wait for something, each with whether it
    stands in an inline assembly block (one of the kernel's own)."""
    found, waits, loads, own = {}, None, False, False
    for line in asm.splitlines():
        m = re.match(r"^(_Z\S+):", line)
        if m:
            waits, loads = (found.setdefault(m.group(1), []) if name in m.group(1) else None), False
        if waits is None:
            continue
        if "#ASMSTART" in line or "#ASMEND" in line:
            own = "#ASMSTART" in line
        s = line.split(";")[0].strip()
        loads = loads or bool(re.match(r"buffer_load_\S+ .*\blds$", s))
        m = re.match(r"s_waitcnt .*vmcnt\((\d+)\)", s)
        if loads and m and int(m.group(1)) < 63:
            waits.append((own, s))
    return found


@pytest.mark.parametrize("src_name,kernel", [(f, k) for f in sorted(KERNELS) for k in KERNELS[f]])
def test_no_compiler_vmcnt_wait_or_scratch(src_name, kernel):
    asm = device_asm(src_name)
    found = _own_waits(asm, kernel)
    assert found
    for fname, waits in found.items():
        assert waits and all(own for own, _ in waits), (fname, [w for own, w in waits if not own][:5])
        assert re.search(rf"\.amdhsa_kernel {re.escape(fname)}\n(?:(?!\.end_amdhsa_kernel).*\n)*?"
                         r"\s*\.amdhsa_private_segment_fixed_size 0\n", asm), f"{fname} uses scratch"


def test_prefill_attention_loop_has_no_compiler_vmcnt_wait():
    funcs = functions(device_asm("attention.hip"))
    bodies = [b for name, b in funcs.items() if "attention_prefill_kernel" in name]
    assert bodies, "attention_prefill_kernel not found"
    for body in bodies:
        first = next(i for i, ins in enumerate(body) if ins.startswith("buffer_load_dwordx4") and ins.endswith("lds"))
        waits = [(i, ins) for i, ins in enumerate(body[first:], first) if ins.startswith("s_waitcnt") and "vmcnt" in ins]
        assert waits, "no vmcnt wait after the first K/V load"
        for i, ins in waits:
            nxt = body[i + 1] if i + 1 < len(body) else ""
            assert nxt == "s_barrier", (i, ins, nxt)
