"""The hand-written waits of the GEMM kernels (csrc/qgemm.hip), checked on the machine code in the built
library, over every path through it. A wave's loads retire in order and `s_waitcnt vmcnt(n)` leaves the
newest n in flight; the kernels count them by hand so that the copies of A rows into LDS two steps ahead
stay in flight across barriers. A count that includes loads the compiler deleted leaves a copy in flight
that the next step reads.

The walk keeps, for a wave, the loads in flight in order and how many barriers each copy has passed.
  * Tile kernels: a copy is read by the other waves one barrier before its own wave reads it, so one in
    flight at its third barrier (`overdue`; the fifth where a step is two halves) must never be followed
    by another operand read.
  * Tile kernels: what a wave reads from LDS is written again by other waves `late` + 1 barriers later at the
    earliest, so its reads have returned when it arrives at the barrier before that.
  * 9- to 64-row kernel (wave-private buffers): at an operand read only the next group's copies may be in
    flight."""
import os
import re
import struct
import subprocess

import pytest

import q38a

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def code_objects(lib):
    """The gfx950 code objects in the library's offload bundles."""
    d = open(lib, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", d):
        at = m.start()
        (n,) = struct.unpack_from("<Q", d, at + 24)
        q = at + 32
        for _ in range(n if n < 16 else 0):
            off, size, tl = struct.unpack_from("<QQQ", d, q)
            name = d[q + 24:q + 24 + tl]
            q += 24 + tl
            if b"gfx950" in name and size:
                yield d[at + off:at + off + size]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled-enough name: [(address, text)]} of the GEMM kernels."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    out = {}
    for i, elf in enumerate(code_objects(q38a.LIB_PATH)):
        if b"qgemm_tile_kernel" not in elf:
            continue
        path = tmp_path_factory.mktemp("isa") / f"{i}.elf"
        path.write_bytes(elf)
        text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
        code = None
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                k = re.search(r"(qgemm_(?:tile|big|small)_kernel)I(\w*?)EEv", m[1])
                code = out.setdefault(k[1] + " " + " ".join(re.findall(r"L[ib](\d+)E", k[2] + "E")), []) if k else None
            elif code is not None and "//" in line:
                ins, rest = line.split("//", 1)
                code.append((int(rest.split(":")[0], 16), ins.strip()))
    assert len(out) == 6 + 3 + 18, sorted(out)
    return out


def walk(code, visit, start):
    """Explores every path: visit(instruction text, state) -> the state after it (None: the path ends)."""
    index = {a: i for i, (a, _) in enumerate(code)}
    seen, todo = set(), [(0, start)]
    while todo:
        i, st = todo.pop()
        while (i, st) not in seen:
            seen.add((i, st))
            addr, ins = code[i]
            op = ins.split()[0]
            if op == "s_endpgm":
                break
            st = visit(ins, st)
            if st is None:
                break
            assert op not in ("s_setpc_b64", "s_swappc_b64"), "an indirect branch"
            if op.startswith(("s_cbranch", "s_branch")):
                off = int(ins.split()[1])
                to = index[addr + 4 + 4 * (off - 65536 if off >= 32768 else off)]
                if op == "s_branch":
                    i = to
                    continue
                todo.append((to, st))
            i += 1


def is_load(ins):
    return ins.startswith(("buffer_load", "global_load", "flat_load", "scratch_load"))


def is_copy(ins):
    return ins.startswith("buffer_load") and ins.endswith(" lds")


def waited(ins, counter):
    """How many operations `s_waitcnt` leaves in flight for the counter, or None."""
    m = re.search(counter + r"\((\d+)\)", ins) if ins.startswith("s_waitcnt") else None
    return int(m[1]) if m else None


@pytest.mark.parametrize("name,overdue", [(f"qgemm_tile_kernel {b} {wm}", 2) for b in (4, 5, 6) for wm in (2, 4)] +
                         [(f"qgemm_big_kernel {b}", 4) for b in (4, 5, 6)])
def test_copies_land_before_they_are_read(kernels, name, overdue):
    late = []

    def visit(ins, st):
        # the loads in flight, oldest first: -1, or the number of barriers a copy has passed; whether
        # a copy was in flight past the barrier that opens it to the readers
        flight, open_ = st
        if is_load(ins):
            flight = (flight + (0 if is_copy(ins) else -1,))[-63:]  # (the counter holds no more: issue stalls)
        n = waited(ins, "vmcnt")
        if n is not None:
            flight = flight[len(flight) - n:] if n else ()
            if n == 0 and waited(ins, "lgkmcnt") == 0:
                open_ = False  # (the full wait after the K loop)
        elif ins.startswith("s_barrier"):
            open_ = open_ or any(f >= overdue for f in flight)
            flight = tuple(f + 1 if f >= 0 else f for f in flight)
        elif ins.startswith("ds_read") and open_:
            late.append(ins)
            return None
        return flight, open_

    walk(kernels[name], visit, ((), False))
    assert not late, f"{len(late)} paths read A rows whose copy may not have landed"


# 128- and 256-row tiles: waves read a buffer in one phase and, in the next, others dequantise or copy into
# it. 256 x 256 tiles: copies and codes go into what was read at least two phases before.
@pytest.mark.parametrize("name,late", [(f"qgemm_tile_kernel {b} {wm}", 0) for b in (4, 5, 6) for wm in (2, 4)] +
                         [(f"qgemm_big_kernel {b}", 1) for b in (4, 5, 6)])
def test_reads_return_before_their_buffer_is_written(kernels, name, late):
    bad = []

    def visit(ins, lds):  # the LDS operations in flight, oldest first: -1, or the barriers a read has passed
        if ins.startswith("ds_"):
            lds += (0 if ins.startswith("ds_read") else -1,)
            assert len(lds) < 64
        n = waited(ins, "lgkmcnt")
        if n is not None:
            lds = lds[len(lds) - n:] if n else ()
        elif ins.startswith("s_barrier"):
            if any(r >= late for r in lds):
                bad.append(ins)
                return None
            lds = tuple(r + 1 if r >= 0 else r for r in lds)
        return lds

    walk(kernels[name], visit, ())
    assert not bad, f"{len(bad)} paths pass a barrier with reads outstanding of a buffer that is written next"


@pytest.mark.parametrize("name", [f"qgemm_small_kernel {b} {rb} {cw} 1" for b in (4, 5, 6) for rb in (1, 2) for cw in (1, 2)])
def test_wave_private_copies_land_before_they_are_read(kernels, name):
    copies = 4 * int(name.split()[2])  # of a group
    late = []

    def visit(ins, flight):
        if is_load(ins):
            flight = (flight + (is_copy(ins),))[-63:]
        n = waited(ins, "vmcnt")
        if n is not None:
            flight = flight[len(flight) - n:] if n else ()
        elif ins.startswith("ds_read") and sum(flight) > copies:
            late.append(ins)
            return None
        return flight

    walk(kernels[name], visit, ())
    assert not late, f"{len(late)} paths read A rows whose copy may not have landed"
