"""Orders that the compiled gfx950 code has to keep and that no output of a
kernel reliably shows, read from the built library."""
import re
import subprocess
from pathlib import Path

import pytest

import mixlab_amd

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The library's gfx950 code objects: (path, symbol table)."""
    lib = Path(mixlab_amd.__file__).parent / "libmixmoe.so"
    if not lib.exists() or not OBJDUMP.exists():
        pytest.skip("needs the built library and llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    (d / "lib.so").symlink_to(lib)
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    return [(co, subprocess.run([OBJDUMP, "-t", co], check=True, capture_output=True,
                                text=True).stdout) for co in sorted(d.glob("lib.so.*gfx950*"))]


def kernels(objects, pattern):
    """{mangled name: instructions} of the kernels whose name matches."""
    found = {}
    for co, syms in objects:
        names = re.findall(rf"(\S*{pattern}\S*Args\w*)$", syms, re.M)
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={','.join(names)}", co],
                              check=True, capture_output=True, text=True).stdout
        for body in re.split(r"\n(?=[0-9a-f]{16} <)", text):
            m = re.match(r"[0-9a-f]{16} <(\S+)>:", body.lstrip())
            if m:
                found[m.group(1)] = [l.split("//")[0].strip() for l in body.splitlines()[1:]]
    assert found, pattern
    return found


def test_ticket_follows_every_waves_release(objects):
    """The one-launch router hands its tokens' results to another workgroup by a
    ticket: before the barrier in front of the ticket's atomic, the waves that
    stored results have written back and waited for their own stores (a barrier
    on this part does not wait for stores to global memory)."""
    code_of = kernels(objects, "route_small_kernel")
    # ...ELi<tokens per workgroup>EEEv14RouteSmallArgs
    tokens = {n: int(re.search(r"Li(\d+)EEEv", n).group(1)) for n in code_of}
    assert set(tokens.values()) == {1, 4}
    for name, code in code_of.items():
        ticket = next(i for i, l in enumerate(code) if l.startswith("global_atomic_add"))
        stores = [i for i, l in enumerate(code[:ticket]) if l.startswith("global_store")]
        assert stores, name
        end = ticket
        if tokens[name] > 1:  # several waves stored: released before the barrier
            end = max(i for i, l in enumerate(code[:ticket]) if l.startswith("s_barrier"))
            assert end > stores[-1], name
        wb = [i for i in range(stores[-1], end) if code[i].startswith("buffer_wbl2 sc1")]
        assert wb, f"{name}: no write-back between the results' stores and the ticket"
        assert any(re.match(r"s_waitcnt vmcnt\(0\)", l) for l in code[wb[-1]:end]), name


def test_combine_reads_picks_with_every_lane_active(objects):
    """The combine of narrow rows reads a token's picks from other lanes'
    registers: those reads stand outside the regions that only some lanes enter
    (a register copied inside one would keep old values in the other lanes)."""
    for name, code in kernels(objects, "combine_wave_kernel").items():
        depth = reads = 0
        for l in code:
            depth += l.startswith("s_and_saveexec_b64")
            depth -= l.startswith("s_or_b64 exec, exec")
            if l.startswith("v_readlane_b32"):
                reads += 1
                assert depth == 0, f"{name}: {l}"
        assert reads > 2, name
