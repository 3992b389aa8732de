"""How the library's kernels are spread over its code objects, which the runtime
loads whole when the first kernel of one is used (no GPU)."""
import os
import re
import struct
import subprocess

import pytest

from test_policies import CSRC, EDITS, POLICIES

LIB = os.path.join(CSRC, "..", "libminiaero_amd.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _kernels():
    """The names of the kernels in each gfx950 code object."""
    data = open(LIB, "rb").read()
    out = []
    for at in (m.start() for m in re.finditer(MAGIC, data)):
        n, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + length]
            p += 24 + length
            if target.endswith(b"gfx950"):
                code = data[at + offset:at + offset + size]
                names = re.findall(rb"\d(k_[a-z0-9_]+?)(?=I|E|P|N)", code)
                walk = re.findall(rb"k_flux_pairI(?:Lb[01]E){4}Lb([01])E", code)
                out.append({x.decode() for x in names} | {"walking " + x.decode() for x in walk})
    return out


def test_forms_on_request_are_an_object_of_their_own():
    """A run that asks neither for the persistent form nor for resident workgroups
    does not load their kernels."""
    on_request = [k for k in _kernels() if k & {"k_steps", "walking 1"}]
    assert len(on_request) == 1 and on_request[0] >= {"k_steps", "walking 1"}
    assert not on_request[0] & {"k_flux", "k_grad", "k_grad_pair", "walking 0"}, sorted(on_request[0])


@pytest.mark.parametrize("what", sorted(EDITS))
def test_forms_on_request_take_the_policies(tmp_path, what):
    """Their unit compiles with a caller's policies,
    which are chosen in solver.hip for it as well."""
    import shutil
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src = tmp_path / "miniaero_amd" / "csrc"
    shutil.copytree(CSRC, src)
    shutil.copytree(os.path.join(CSRC, "..", "..", "include"), tmp_path / "include")
    text = (src / "physics.hpp").read_text()
    at = text.rindex("}  // namespace ma")
    (src / "physics.hpp").write_text(text[:at] + POLICIES + text[at:])
    text = (src / "solver.hip").read_text()
    for old, new in EDITS[what]:
        text = text.replace(old, new)
    (src / "solver.hip").write_text(text)
    r = subprocess.run([hipcc, "-fsyntax-only", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                        "--offload-arch=gfx950", "--offload-device-only", str(src / "steps.hip")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
