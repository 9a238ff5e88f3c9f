"""The one-launch router hands its tokens' results to another workgroup by a
ticket.  Read from the built gfx950 code: before the barrier in front of the
ticket's atomic, the waves that stored results have written back and waited for
their own stores (a barrier on this part does not wait for stores to global
memory)."""
import re
import subprocess
from pathlib import Path

import pytest

import mixlab_amd

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    lib = Path(mixlab_amd.__file__).parent / "libmixmoe.so"
    if not lib.exists() or not OBJDUMP.exists():
        pytest.skip("needs the built library and llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    (d / "lib.so").symlink_to(lib)
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    found = {}
    for co in sorted(d.glob("lib.so.*gfx950*")):
        syms = subprocess.run([OBJDUMP, "-t", co], check=True, capture_output=True, text=True).stdout
        names = re.findall(r"(\S*route_small_kernel\S*Args)$", syms, re.M)
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={','.join(names)}", co],
                              check=True, capture_output=True, text=True).stdout
        for body in re.split(r"\n(?=[0-9a-f]{16} <)", text):
            m = re.match(r"[0-9a-f]{16} <(\S+)>:", body.lstrip())
            if m:
                found[m.group(1)] = [l.split("//")[0].strip() for l in body.splitlines()[1:]]
    assert found
    return found


def test_ticket_follows_every_waves_release(kernels):
    # ...ELi<tokens per workgroup>EEEv14RouteSmallArgs
    tokens = {n: int(re.search(r"Li(\d+)EEEv", n).group(1)) for n in kernels}
    assert set(tokens.values()) == {1, 4}
    for name, code in kernels.items():
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
