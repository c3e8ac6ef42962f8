"""The library's gfx950 code, for tests that look at what the compiler made of a kernel (built here from source)."""
import re
import struct
import subprocess

LLVM = "/opt/rocm/llvm/bin/"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib, tmp_path):
    """The gfx950 code objects that the library embeds, one per source file with kernels, as files."""
    fat = tmp_path / "fatbin"
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", lib, "/dev/null"], check=True)
    data, at, files = fat.read_bytes(), 0, []
    while (at := data.find(MAGIC, at)) >= 0:
        n, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if "gfx950" in triple and size:
                files.append(tmp_path / f"co{len(files)}")
                files[-1].write_bytes(data[at + offset:at + offset + size])
        at += len(MAGIC)
    return files


def kernels(code_object):
    """name -> [(address, mnemonic, operands, branch target or None)] in program order."""
    text = subprocess.run([LLVM + "llvm-objdump", "-d", "--demangle", "--mcpu=gfx950", str(code_object)], check=True,
                          capture_output=True, text=True).stdout
    out, body = {}, None
    for line in text.splitlines():
        if m := re.match(r"^[0-9a-f]+ <(.*)>:$", line):
            body = out.setdefault(m.group(1), [])
            base = int(line.split(" ", 1)[0], 16)
        elif body is not None and "//" in line:
            asm, note = line.split("//", 1)
            op, _, args = asm.strip().partition(" ")
            target = re.search(r"<.*\+0x([0-9a-f]+)>\s*$", note) if op.startswith(("s_cbranch", "s_branch")) else None
            body.append((int(note.split(":")[0], 16), op, args.strip(), base + int(target.group(1), 16) if target else None))
    return out


def loads_under_way_at_barriers(code):
    """Largest number of loads into LDS that may still be under way at each barrier, over all paths: address -> count.

    Vector-memory instructions finish in the order of their issue, and `s_waitcnt vmcnt(n)` waits until n are left: the
    state is the list of those under way, oldest first, each one a load into LDS or not."""
    index = {a: i for i, (a, *_) in enumerate(code)}
    seen, todo, at_barrier = set(), [(0, ())], {}
    while todo:
        i, flight = todo.pop()
        while i < len(code) and (i, flight) not in seen:
            seen.add((i, flight))
            address, op, args, target = code[i]
            if op.startswith(("buffer_", "global_", "flat_", "scratch_")) and not op.startswith(("buffer_wbl2", "buffer_inv")):
                flight = (flight + (bool(re.search(r"\blds\b", args)),))[-64:]
            elif op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", args)):
                n = int(m.group(1))
                flight = flight[len(flight) - n:] if n < len(flight) else flight
                if n == 0:
                    flight = ()
            elif op == "s_barrier":
                at_barrier[address] = max(at_barrier.get(address, 0), sum(flight))
            elif op == "s_endpgm":
                break
            # what lies before the oldest load into LDS cannot matter any more
            while flight and not flight[0]:
                flight = flight[1:]
            if target is not None:
                if op == "s_branch":
                    i = index[target]
                    continue
                todo.append((index[target], flight))
            i += 1
    return at_barrier


def registers(code_object):
    """mangled name -> vector registers (both kinds) of each kernel."""
    notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(code_object)], check=True, capture_output=True, text=True).stdout
    found = re.findall(r"\.name: +(\S+)\n(?:(?!\.name:).)*?\.vgpr_count: +(\d+)", notes, re.S)
    return {n: int(r) for n, r in found}
