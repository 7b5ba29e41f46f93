"""What the compiler makes of the kernels, read from its assembly: no variable that should be a register ends up in memory.
Without a GPU."""
import concurrent.futures
import glob
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build_module():
    spec = importlib.util.spec_from_file_location("build_flags", os.path.join(ROOT, "dcgan-cuda_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """{source: assembly text}"""
    b = build_module()
    if not os.path.exists(b.HIPCC):
        pytest.skip("hipcc not found")
    out = tmp_path_factory.mktemp("asm")

    def one(src):
        name = os.path.basename(src)
        s = str(out / (name + ".s"))
        subprocess.run([b.HIPCC] + b.HIPFLAGS + ["--cuda-device-only", "-S", src, "-o", s], check=True, capture_output=True)
        return name, open(s).read()
    with concurrent.futures.ThreadPoolExecutor(8) as ex:
        return dict(ex.map(one, sorted(glob.glob(os.path.join(b.CSRC, "*.hip")))))


def kernels(text):
    """(name, descriptor directives as a dict) of every kernel"""
    for m in re.finditer(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", text, re.S):
        yield m.group(1), dict(re.findall(r"\.amdhsa_(\S+) (\S+)", m.group(2)))


def test_no_variable_in_lds(assembly):
    """A local variable that the compiler cannot keep in a register and moves to LDS is indexed by the workgroup's extents, which
    it reads from the dispatch packet: the one use of that pointer here, no kernel asks for its extents."""
    count = 0
    for src, text in assembly.items():
        for name, d in kernels(text):
            count += 1
            assert d["user_sgpr_dispatch_ptr"] == "0", (src, name)
    assert count > 100


def test_no_spills(assembly):
    """No kernel keeps registers in memory."""
    for src, text in assembly.items():
        spills = dict(zip(re.findall(r"\.symbol:\s*(\S+)", text), re.findall(r"\.vgpr_spill_count:\s*(\d+)", text)))
        for name, d in kernels(text):
            assert d["private_segment_fixed_size"] == "0" and spills.get(name + ".kd", spills.get("'" + name + ".kd'")) == "0", (src, name)


def test_no_loop_around_a_load(assembly):
    """The address of a buffer is the same for all lanes: where the compiler cannot tell, it puts a loop over the lanes around the
    load, which ends in a branch on the lanes left."""
    for src, text in assembly.items():
        for name, body in re.findall(r"^(\S*conv_igemm_fast\S*):(.*?)s_endpgm", text, re.S | re.M):
            lines = [l.split()[0] for l in body.split("\n") if l.startswith("\t") and l.split()]
            loops = sum(l.startswith("buffer_load") and "s_cbranch_execnz" in lines[i:i + 4] for i, l in enumerate(lines))
            assert loops == 0, (src, name, loops)


def test_no_second_copy_of_the_input_gradient(assembly):
    """The general kernel has a variant for filters of fewer elements than a wide load reads (the last template argument). The input gradient has no such load, and
    a variant would be a copy of the kernel that nothing launches."""
    for src, wanted in (("conv_fwd.hip", 4), ("conv_dk.hip", 4), ("conv_dx.hip", 0)):       # one per tile shape
        names = [name for name, _ in kernels(assembly[src]) if re.search(r"conv_igemmI\w*Li1ELb0EEE", name)]
        assert len(names) == wanted, (src, names)
