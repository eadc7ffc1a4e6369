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
