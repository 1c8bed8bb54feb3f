"""The waits of the tiles with weight operands in registers (csrc/q4_gemm_wide.hip), counted in the code that was built.

Their activations are written into LDS by the loads, a row tile per reduction step, by all four wavefronts; a barrier hands a
tile over, and before it every wavefront waits until only so many of its youngest requests are left.  That count is right only
while the requests it passes over exist: one to a register that nothing reads any more is deleted by the compiler.  Here every
path through a kernel is followed with the queue of its requests: behind the j-th barrier of a pipeline nothing of the tiles
0 .. j may be on its way.  (An output shows such a fault only when a load happens to be late.)"""
import os
import re
import struct
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "alpaca_lora_4bit_amd", "libq4gptq.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNELS = {f"_ZN2q4{len(name)}{name}ILi{tm}ELb{fwd}EEEvNS_{args}E": (tm, name)
           for name, args in (("gemm_wide_kernel", "8GemmArgs"), ("gemm_wide_group_kernel", "13GemmGroupArgs"))
           for tm, fwd in ((8, 1), (4, 1), (8, 0))}


def code_objects(data):
    """The gfx950 code objects of the library's offload bundles."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", -1
    while (at := data.find(magic, at + 1)) >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, pos - 8)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + n]:
                yield data[at + off:at + off + size]
            pos += 24 + n


def parse(text):
    """[(address, mnemonic, operands, target address or None)] of a disassembled function"""
    out = []
    for line in text.splitlines():
        m = re.match(r"\s+(\S+)(.*?)//\s*([0-9A-F]{8,}):", line)
        if not m:
            continue
        addr, target = int(m.group(3), 16), None
        if m.group(1).startswith(("s_cbranch", "s_branch")):
            jump = int(m.group(2).split()[0])
            target = addr + 4 + 4 * (jump - 65536 if jump >= 32768 else jump)
        out.append((addr, m.group(1), m.group(2), target))
    return out


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler for the built library")
    with open(LIB, "rb") as f:
        data = f.read()
    found = {}
    for i, blob in enumerate(code_objects(data)):
        names = [k for k in KERNELS if k.encode() in blob]
        if not names:
            continue
        path = tmp_path_factory.mktemp("obj") / f"{i}.o"
        path.write_bytes(blob)
        text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(names), str(path)], check=True,
                              capture_output=True, text=True).stdout
        parts = re.split(r"^[0-9a-f]+ <(\S+)>:\n", text, flags=re.M)
        found.update({parts[j]: parse(parts[j + 1]) for j in range(1, len(parts), 2)})
    return found


def is_request(op):
    return re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", op) is not None


def late_tiles(code, tm):
    """(barrier address, tile, requests of it that may still be on their way) wherever a path breaks the rule above"""
    index = {ins[0]: i for i, ins in enumerate(code)}
    first = next(i for i, ins in enumerate(code) if ins[1].startswith("buffer_load") and " lds" in ins[2])
    assert sum(ins[1] == "s_barrier" for ins in code[first:]) >= 6
    faults, seen = set(), set()
    # queue: tile of each request to LDS relative to the barriers passed, None for other requests, oldest first
    todo = [(first, (), 0, 0)]                          # instruction, queue, barriers passed - tiles requested in full, requests of the next tile
    while todo:
        i, queue, ahead, part = todo.pop()
        while i < len(code):
            addr, op, args, target = code[i]
            if op == "s_endpgm" or "store" in op:       # the pipeline is over
                break
            if is_request(op):
                if " lds" in args:
                    queue += (-ahead,)
                    part += 1
                    if part == tm:
                        ahead, part = ahead - 1, 0
                else:
                    queue += (None,)
                queue = queue[-64:]                     # the counter waits for anything older by itself
            elif op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", args)):
                n = int(m.group(1))
                queue = queue[len(queue) - n:] if n < len(queue) and n else queue if n else ()
            elif op == "s_barrier":
                late = [t for t in queue if t is not None and t <= 0]
                faults.update((addr, t, late.count(t)) for t in late)
                queue = tuple(None if t is None else t - 1 for t in queue)
                ahead += 1
            if target is not None:
                state = (target, queue, ahead, part)
                if state not in seen and index.get(target, -1) >= first:       # a branch to in front of it: the next layer starts over
                    seen.add(state)
                    todo.append((index[target], queue, ahead, part))
                if op == "s_branch":
                    break
            i += 1
    return faults


@pytest.mark.parametrize("kernel", sorted(KERNELS))
def test_no_tile_is_handed_over_before_it_has_landed(listings, kernel):
    tm, _ = KERNELS[kernel]
    assert late_tiles(listings[kernel], tm) == set()
