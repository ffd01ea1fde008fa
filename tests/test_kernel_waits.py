"""Waits in the built code of the attention kernels that copy tiles to LDS while they work on others (compiled here, no device needed)."""
import os
import re
import subprocess

import pytest
from conftest import ROOT

CSRC = os.path.join(ROOT, "moondream-zig_amd", "csrc")


@pytest.fixture(scope="module")
def copying_loops(tmp_path_factory):
    """(file, kernel) -> the first loop of the kernel that copies tiles to LDS, as lines of assembly"""
    flags = subprocess.run(["make", "-s", "-C", CSRC, "--eval", "flags: ; @echo $(HIPCC) $(HIPFLAGS)", "flags"], check=True, capture_output=True, text=True).stdout.split()
    out = {}
    for name in ("attn_prefill", "attn_window"):
        path = tmp_path_factory.mktemp(name) / "out.s"
        subprocess.run([*flags, "-w", "--offload-device-only", "-S", f"{name}.hip", "-o", str(path)], check=True, cwd=CSRC, capture_output=True)
        for kernel, body in re.findall(r"^(_Z\w+):(.*?)^\.Lfunc_end", path.read_text(), re.S | re.M):
            blocks = re.split(r"^(?=\.LBB\w+:|; %bb\.\d+:)", body, flags=re.M)
            headers = [re.match(r"\.L(BB\w+):", b).group(1) for b in blocks if re.match(r"\.LBB\w+:.*Loop Header", b)]
            for header in headers:
                loop = "".join(b for b in blocks if b.startswith(f".L{header}:") or re.match(rf".*in Loop: Header={header}\b", b))
                if re.search(r"buffer_load_dwordx4 .* lds$", loop, re.M):
                    out[name, kernel] = loop.splitlines()
                    break
    return out


def test_the_kernels_are_there(copying_loops):
    names = " ".join(kernel for _, kernel in copying_loops)
    assert len(re.findall(r"window_attn_shared_kernel", names)) == 4 and len(re.findall(r"flash_attn(?:64|96)_kernel", names)) == 3


def test_no_wait_for_copies_but_those_in_the_source(copying_loops):
    """A copy is under way while the tile before it is worked on.  The compiler does not see what the source waits for: loads that it still counts as under way
    ahead of the loop become a wait in the loop, and with it for the copies issued last."""
    for kernel, loop in copying_loops.items():
        inside, found = False, []
        for line in loop:
            inside = inside and "#ASMEND" not in line or "#ASMSTART" in line
            if not inside and re.search(r"s_waitcnt.*vmcnt", line):
                found.append(line.strip())
        assert not found, (kernel, found)


def test_tiles_are_handed_over_behind_waits_of_the_source(copying_loops):
    """Behind a shared tile's barrier others copy over the tile before: reads of it must have returned, whatever the compiler puts between them and the barrier."""
    shared = {kernel: [i for i, line in enumerate(loop) if "s_barrier" in line] for kernel, loop in copying_loops.items()}
    assert sum(map(bool, shared.values())) == 5
    for kernel, barriers in shared.items():
        for i in barriers:
            lines = [line.split(";")[0].split() for line in copying_loops[kernel][:i] if line.split(";")[0].strip()]
            assert lines[-1] == ["s_waitcnt", "vmcnt(0)", "lgkmcnt(0)"], (kernel, lines[-1])
