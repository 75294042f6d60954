"""What the compiler made of kernels whose speed hangs on it, read from the
built library's own gfx950 code objects: no scratch memory in the Widom finish
kernels (every launch would set it up), no ragged-workgroup set-up in the pair
kernels (the workgroup size is a constant there)."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    from graspa_amd import engine
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no LLVM tools")
    if not os.path.exists(engine.LIB_PATH):
        pytest.skip("the library is not built")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(engine.LIB_PATH, d / "lib.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True,
                   stdout=subprocess.DEVNULL)
    out = sorted(str(d / f) for f in os.listdir(d) if f.endswith("gfx950"))
    assert out
    return out


def _run(tool, *args):
    return subprocess.run([os.path.join(LLVM, tool), *args], check=True, capture_output=True, text=True).stdout


def test_finish_kernels_have_no_scratch(code_objects):
    scratch = {}
    for f in code_objects:
        for k in re.split(r"\n  - \.agpr_count", _run("llvm-readelf", "--notes", f))[1:]:
            name = re.search(r"\.name: +(_Z\w+)", k).group(1)
            scratch[name] = int(re.search(r"\.private_segment_fixed_size: (\d+)", k).group(1))
    finish = {n: s for n, s in scratch.items() if "widom_finish" in n}
    assert len(finish) == 5
    assert not any(finish.values()), finish


def test_pair_kernels_do_not_read_the_workgroup_size(code_objects):
    seen, bad, name = set(), [], ""
    for f in code_objects:
        for line in _run("llvm-objdump", "-d", "--no-show-raw-insn", f).splitlines():
            m = re.match(r"[0-9a-f]{16} <(\w+)>:", line)
            if m:
                name = m.group(1)
                if "widom_eval" in name:
                    seen.add(name)
            elif "widom_eval" in name and "global_load_ushort" in line:
                bad.append(name)
    assert len(seen) == 64
    assert not bad
