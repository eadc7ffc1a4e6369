"""Waits of a kernel that places its own barriers, in the code that was built (no GPU)."""
import os
import re
import subprocess

from decdec_amd import _lib

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def _kernels(library, name, folder):
    """Instructions of the kernels whose symbol holds `name`, by symbol."""
    link = os.path.join(folder, "library.so")
    os.symlink(library, link)
    subprocess.run([OBJDUMP, "--offloading", link], check=True, stdout=subprocess.DEVNULL, cwd=folder)
    found = {}
    for image in sorted(os.listdir(folder)):
        path = os.path.join(folder, image)
        if not image.endswith("gfx950") or name.encode() not in open(path, "rb").read():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", path], check=True, stdout=subprocess.PIPE, text=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            symbol, _, code = part.partition(">:\n")
            if name in symbol:
                found[symbol] = [line.split("//")[0].strip() for line in code.splitlines() if line.startswith("\t")]
    return found


def test_wide_tiles_read_a_buffer_to_the_end_before_it_is_copied_to_again(tmp_path):
    """Behind the barrier of a packet every wave requests copies into the buffer that the packet before was read from: all of a wave's reads
    have to be there when it comes to the barrier.  (The products that use them may follow behind it, and did.)"""
    kernels = _kernels(_lib.LIB_PATH, "qgemm_wide_kernel", str(tmp_path))
    assert len(kernels) >= 10
    for symbol, code in kernels.items():
        barriers = [i for i, line in enumerate(code) if line.startswith("s_barrier")]
        assert barriers, symbol
        for at in barriers:
            before = next(line for line in reversed(code[:at]) if line.startswith("ds_") or "lgkmcnt(0)" in line or line.startswith(("s_cbranch", "s_branch")))
            assert "lgkmcnt(0)" in before, f"{symbol}: `{before}` before a barrier"


def test_copies_into_lds_come_behind_every_read_of_what_they_replace(tmp_path):
    """The same for tiles of 128 tokens, whose ranges of channels also meet at barriers that nothing has to be there for: between a wave's last read and
    its next copy it has waited for its reads, and then for the other waves."""
    kernels = _kernels(_lib.LIB_PATH, "qgemm_kernel", str(tmp_path))
    assert len(kernels) >= 100
    for symbol, code in kernels.items():
        copies = 0
        waited, met = True, True                           # nothing read yet
        for line in code:
            if line.startswith("ds_read"):
                waited = met = False
            elif line.startswith("s_waitcnt") and "lgkmcnt(0)" in line:
                waited = True
            elif line.startswith("s_barrier"):
                met = met or waited
            elif line.startswith("global_load_lds"):
                copies += 1
                assert met, f"{symbol}: a copy into LDS ahead of the barrier"
        assert copies, symbol


def _addressed(library, name, folder):
    """(address, instruction, address it may go to) of the kernels whose symbol holds `name`, by symbol."""
    link = os.path.join(folder, "library.so")
    os.symlink(library, link)
    subprocess.run([OBJDUMP, "--offloading", link], check=True, stdout=subprocess.DEVNULL, cwd=folder)
    found = {}
    for image in sorted(os.listdir(folder)):
        path = os.path.join(folder, image)
        if not image.endswith("gfx950") or name.encode() not in open(path, "rb").read():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", path], check=True, stdout=subprocess.PIPE, text=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            symbol, _, code = part.partition(">:\n")
            if name not in symbol:
                continue
            lines = [re.match(r"\t(.*?)\s*// ([0-9A-F]+):", line) for line in code.splitlines() if line.startswith("\t")]
            lines = [(int(m.group(2), 16), m.group(1)) for m in lines if m]             # what is between kernels has no address
            follows = [(at, line, following[0]) for (at, line), following in zip(lines, lines[1:] + [(None, None)])]
            code = []
            for at, line, following in follows:
                goes = None
                if line.startswith(("s_branch", "s_cbranch")):
                    words = int(line.split()[-1])
                    goes = at + 4 + 4 * (words - 65536 if words > 32767 else words)
                code.append((at, line, goes))
            found[symbol] = code
    return found


def _early_reads(code, tasks, first_wait, first_packets):
    """What a wave of `code` does with a packet's activations that may not be there, or None: along every way through the kernel, with `tasks` copies a packet.

    Requests to memory return in order: a wait for N leaves the last N.  A packet's wait is the one that also waits for LDS.  Behind it, at the barrier, none of that packet's
    copies may be out, and its reads follow.  `first_wait` is the number of a wait that only the first `first_packets` packets take."""
    index = {at: i for i, (at, _, _) in enumerate(code)}
    # place, packets waited for (up to 3), requests that are out (a copy: packets ahead of the one that is read; others None), copies begun, wait without barrier
    start = (0, 0, (), (0, 0), False)
    seen, todo, packets = {start}, [start], 0
    while todo:
        i, waited, out, (group, copied), armed = todo.pop()
        at, line, goes = code[i]
        op, ways = line.split()[0], [i + 1]
        if op == "s_endpgm":
            continue
        if op.startswith("global_load_lds"):
            out += (group,)
            copied += 1
            if copied == tasks:
                group, copied = group + 1, 0
        elif op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            out += (None,)
        elif op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", line)
            if m:
                out = out[len(out) - min(len(out), int(m.group(1))):]
                if "lgkmcnt(0)" in line:
                    if int(m.group(1)) == first_wait and waited >= first_packets:
                        continue                           # not a way that is taken
                    if waited > 0:                         # the next packet
                        out, group = tuple(None if c is None else c - 1 for c in out), group - 1
                    waited, armed, packets = min(waited + 1, 3), True, packets + 1
        elif op == "s_barrier" and armed:
            if any(c is not None and c <= 0 for c in out):
                return f"{at:x}: copies of a packet are out at its barrier: {out}"
            armed = False
        elif op.startswith("ds_read") and armed:
            return f"{at:x}: a read ahead of the barrier"
        if goes is not None:
            # lanes are never all off where a branch looks at that to go around the other way
            ways = [index[goes]] if op in ("s_branch", "s_cbranch_execnz") else [i + 1, index[goes]]
        for way in ways:
            state = (way, waited, out[-63:], (group, copied), armed)
            if state not in seen:
                seen.add(state)
                todo.append(state)
    return None if packets >= 8 else "no packets were found"


def _packet_numbers(symbol):
    """Copies of a packet and the first packets' wait, from the template arguments."""
    fmt, bits, _, mt, flag = (int(v) for v in re.search(r"qgemm_kernelILi(\d)ELi(\d)ELi(\d)ELi(\d)ELb(\d)E", symbol).groups())
    tasks, three = 4 * mt // (4 if mt >= 3 else 2), mt <= 6
    words = 2 * (2 if flag else 4) * bits if fmt == 0 else 4 * 2 * bits
    return tasks, words + (tasks if three else 0), 2 if three else 1


def test_a_packets_copies_are_there_when_it_is_read(tmp_path):
    """The waits of the tiles of 128 tokens count what was asked for behind a packet's copies: as many requests as they count have to stand there, on every way through
    the code that was built."""
    kernels = _addressed(_lib.LIB_PATH, "qgemm_kernel", str(tmp_path))
    assert len(kernels) >= 100
    for symbol, code in kernels.items():
        assert _early_reads(code, *_packet_numbers(symbol)) is None, (symbol, _early_reads(code, *_packet_numbers(symbol)))
    # a word's request fewer, or waits that leave one more, are seen
    symbol = min(kernels)
    code, numbers = kernels[symbol], _packet_numbers(symbol)
    loads = [i for i, (_, line, _) in enumerate(code) if line.startswith("global_load_dword")]
    fewer = [(at, "s_nop 0" if i == loads[len(loads) // 2] else line, goes) for i, (at, line, goes) in enumerate(code)]
    weaker = [(at, re.sub(r"\d+", lambda m: str(int(m.group()) + 1), line, count=1) if line.startswith("s_waitcnt vmcnt") and line.endswith("lgkmcnt(0)") else line, goes)
              for at, line, goes in code]
    assert _early_reads(fewer, *numbers) and _early_reads(weaker, numbers[0], numbers[1] + 1, numbers[2])


def test_a_wide_tiles_copies_are_there_when_they_are_read(tmp_path):
    """The same for tiles of 256 tokens, packet by packet between barriers: the second waves copy ahead of a packet's words and wait behind its products, the first copy behind
    the products before and wait behind the words.  Either wait counts the packet's words, of which at least as many are requested behind either copy."""
    kernels = _kernels(_lib.LIB_PATH, "qgemm_wide_kernel", str(tmp_path))
    for symbol, code in kernels.items():
        fmt, bits, _, mt = (int(v) for v in re.search(r"qgemm_wide_kernelILi(\d)ELi(\d)ELi(\d)ELi(\d+)E", symbol).groups())
        rounds = 16 * mt // 32                             # copies of a wave and packet
        kinds = {"global_load_lds": "C", "global_load": "L", "s_barrier": "B", "ds_read": "R"}
        text = "".join(next((k for start, k in kinds.items() if line.startswith(start)), f"[{line.split('(')[1].split(')')[0]}]" if line == f"s_waitcnt vmcnt({2 * bits})" else "")
                       for line in code)
        wait = rf"\[{2 * bits}\]"
        packets = re.findall(rf"C{{{rounds}}}((?:L|{wait})*{wait})B((?:R|{wait})+)C{{{rounds}}}(?:{wait})+B", text)
        assert len(packets) == 4, (symbol, text)
        for words, reads in packets:
            assert words.count("L") >= 2 * bits and reads.count("R") == 4 * mt, (symbol, text)
