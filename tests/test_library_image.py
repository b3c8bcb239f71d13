"""What the built library says about its kernels (the gfx950 code objects' own metadata), where a kernel's code counts on it."""
import os
import re
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
CSRC = os.path.join(ROOT, "project-maya_amd", "csrc")


def code_objects(path):
    """The gfx950 code objects in a library's offload bundles."""
    d, at = open(path, "rb").read(), 0
    while (b := d.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        n, = struct.unpack_from("<Q", d, b + 24)
        at = b + 32
        for _ in range(n):
            off, size, name_len = struct.unpack_from("<QQQ", d, at)
            name = d[at + 24:at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name:
                yield d[b + off:b + off + size]


def kernels(path):
    """name -> metadata of every gfx950 kernel in a library's offload bundles."""
    return {n: k for e in code_objects(path) for n, k in code_object_kernels(e)}


def instructions(path, names, tmp_path):
    """name -> the instructions of the kernels `names`, as the assembler writes them."""
    found = {}
    for i, e in enumerate(code_objects(path)):
        co = tmp_path / ("%d.co" % i)
        co.write_bytes(e)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--disassemble-symbols=" + ",".join(names), str(co)],
                              capture_output=True, text=True, check=True).stdout
        for part in re.split(r"^(?=(?:[0-9a-f]+ )?<\S+>:$)", text, flags=re.M)[1:]:
            head, *lines = part.splitlines()
            found[re.search(r"<(\S+)>:", head).group(1)] = [l.split("//")[0].strip() for l in lines if l.strip()]
    return found


def code_object_kernels(e):
    sections, = struct.unpack_from("<Q", e, 40)
    entry, count = struct.unpack_from("<HH", e, 58)
    for i in range(count):
        _, kind, _, _, at, size = struct.unpack_from("<IIQQQQ", e, sections + i * entry)
        end = at + size
        while kind == 7 and at < end:   # SHT_NOTE
            name_size, desc_size, note = struct.unpack_from("<III", e, at)
            desc = at + 12 + (name_size + 3) // 4 * 4
            at = desc + (desc_size + 3) // 4 * 4
            if note == 32:              # NT_AMDGPU_METADATA
                yield from ((k[".name"], k) for k in msgpack.unpackb(e[desc:desc + desc_size], strict_map_key=False)["amdhsa.kernels"])


def built():
    lib = os.path.join(ROOT, "project-maya_amd", "libmaya_moe.so")
    if not os.path.exists(lib):
        from maya_amd import build
        build.build()
    return lib


def test_kernels_of_rows_a_wave_spill_nothing():
    """Register limits are chosen so that the loops over weight rows keep everything in registers."""
    got = {n: k for n, k in kernels(built()).items() if "down_q4k_pos_kernel" in n or "gate_up_iq2xxs_pos_kernel" in n}
    assert len(got) >= 10
    for n, k in got.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, n


def test_the_iq2s_prompt_kernels_have_no_lds_but_their_array():
    """Their tables' look-ups count LDS addresses from 0: a second object there is refused at the first call, and seen here first."""
    lds = int(re.search(r"\bkIqLdsBytes = (\d+);", open(os.path.join(CSRC, "maya_prefill_iq2s.hpp")).read()).group(1))
    got = {n: k for n, k in kernels(built()).items() if "prefill_iq2s_kernel" in n}
    assert len(got) == 2
    for n, k in got.items():
        assert k[".group_segment_fixed_size"] == lds, n
    few = {n: k for n, k in kernels(built()).items() if "prefill_iq2s_few_kernel" in n}   # (the same tables, a shorter ring)
    assert len(few) == 2 and len({k[".group_segment_fixed_size"] for k in few.values()}) == 1
    assert all(k[".group_segment_fixed_size"] <= 160 * 1024 // 3 and k[".private_segment_fixed_size"] == 0 for k in few.values())


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_one_token_of_iq2s_waits_for_nothing_before_its_first_loads(tmp_path):
    """What the router is given arrives in registers with the dispatch: a wait in front of the first load is a trip to memory that every
    workgroup makes first.  (In front of the body stands a prologue that loads and waits, for firmware that does not preload.)"""
    names = [n for n in kernels(built()) if re.search(r"gate_up_iq2s_tiles_kernelILi\dELi\dELi[48]ELb0E", n)]
    assert len(names) == 14
    for n, code in instructions(built(), names, tmp_path).items():
        body = code[next(i for i, c in enumerate(code) if c.startswith("s_branch")) + 1:]
        first = next(i for i, c in enumerate(body) if c.startswith("global_load"))
        assert not [c for c in body[:first] if c.startswith("s_waitcnt")], n


def test_one_token_heads_leave_seven_waves_a_simd():
    """Q4_K rows that fill their lanes (16 rows a workgroup) and IQ1_S rows of three waves and more, the layer's head in the launch: 72
    registers at most, the form of several tokens has 75."""
    got = {n: k for n, k in kernels(built()).items()
           if re.search(r"gate_up_q4k_pos_kernelILi\dELi16ELi6ELb1ELb0ELi4ELb0E|gate_up_iq1s_pos_kernelILi[3-8]ELi16ELi6ELb[01]ELi[48]ELb0E", n)}
    assert len(got) == 7 + 18
    for n, k in got.items():
        assert k[".vgpr_count"] <= 72 and k[".private_segment_fixed_size"] == 0, n


def test_the_iq2s_tile_walk_holds_the_workgroups_it_is_launched_with():
    """Eight of two waves a compute unit, three of more, whichever form the layer's head has: 512 registers a lane of a SIMD in blocks
    of 8, 160 KB of LDS."""
    got = {n: k for n, k in kernels(built()).items() if "gate_up_iq2s_tiles_kernel" in n}
    assert len(got) == 7 * 5
    for n, k in got.items():
        waves = int(re.search(r"kernelILi(\d)E", n).group(1))
        wgs = 8 if waves == 2 else 3
        assert wgs * k[".group_segment_fixed_size"] <= 160 * 1024, n
        assert -(-wgs * waves // 4) <= 512 // (-(-k[".vgpr_count"] // 8) * 8), n
