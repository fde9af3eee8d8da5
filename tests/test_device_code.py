"""What the kernels ask of the compiler, read from the unoptimised code of the device sources: it
holds whatever a compiler's passes make of it, where a run shows today's build only."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "vina-cuda_amd", "csrc")


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    """Mangled name -> body, of kernels.hip as the front end emits it."""
    out = str(tmp_path_factory.mktemp("ir") / "kernels.ll")
    subprocess.check_call([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-emit-llvm", "-S",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Xclang", "-disable-llvm-passes",
                           "-w", "-o", out, os.path.join(CSRC, "kernels.hip")])
    with open(out) as f:
        return {m.group(1): m.group(2) for m in re.finditer(r"^define [^@]*@(\S+?)\(.*?\{$(.*?)^\}", f.read(), re.M | re.S)}


def calls(body, *names):
    """The calls of a body to any of the named functions, in order."""
    found = re.findall(r"call [^@]*@(\S+?)\(", body)
    return [n for f in found for n in names if re.search(r"\d%s[A-Z]" % n, f)]


def test_rows_of_a_wide_chain_update_a_node_in_turn(functions):
    """A node whose atoms lie in several rows of 16 lanes: each row's update is fenced from the next."""
    wide = [b for n, b in functions.items() if re.match(r"_ZN3vdk10eval_derivILi16ELb1", n)]
    assert len(wide) == 3   # the three modes
    for body in wide:
        assert calls(body, "add_to_node", "wave_sync") == ["add_to_node", "wave_sync"]


def test_exchange_row_of_a_wide_chain_is_fenced(functions):
    """Slots written by all lanes, read by the lanes that own their atoms, written again."""
    body, = [b for n, b in functions.items() if n.startswith("_ZN3vdk15pair_terms_wide")]
    assert re.search(r"call [^@]*@_ZN3vdk9wave_sync", body)
    order = re.findall(r"call [^@]*@(_ZN3vdk9wave_sync|_ZZN3vdk15pair_terms_wide\S*?RK?15HIP_vector_typeIfLj4EES9_IjLj2EE)", body)
    assert ["sync" if "wave_sync" in o else "take" for o in order] == ["sync", "take", "take", "sync"]


def test_wave_sync_is_a_fence_and_a_barrier(functions):
    for ns in ("3vdk", "3vdr"):
        body, = [b for n, b in functions.items() if n.startswith("_ZN%s9wave_syncEv" % ns)]
        assert 'fence syncscope("wavefront") acq_rel' in body and "@llvm.amdgcn.wave.barrier" in body


def test_half_rows_of_the_map_table_are_read_at_their_alignment(functions):
    """Half 1 of a 48-byte row lies at a multiple of 8 bytes, so no read of a half may promise 16."""
    body, = [b for n, b in functions.items() if re.match(r"_ZN12_GLOBAL__N_19load_half", n)]
    reads = re.findall(r"load <4 x float>, ptr \S+, align (\d+)", body)
    copies = re.findall(r"@llvm.memcpy\S*\(ptr align \d+ \S+, ptr align (\d+)", body)
    assert reads + copies and all(int(a) <= 8 for a in reads + copies)
    kernels = [b for n, b in functions.items() if re.match(r"_ZN12_GLOBAL__N_114vd_grid_kernel", n)]
    assert kernels and all(calls(b, "load_half") == ["load_half"] for b in kernels)


def test_every_compiled_form_is_launched(functions):
    """Dense BFGS takes three waves per SIMD on 64 lanes only; the map kernel has two forms."""
    names = [m.groups() for m in (re.match(r"_ZN12_GLOBAL__N_112vd_mc_kernelILi(\d+)ELi(\d)ELi(\d)E", n) for n in functions) if m]
    assert {n for n in names if n[1] == "0"} == {("64", "0", "2"), ("32", "0", "2"), ("16", "0", "2"), ("64", "0", "3")}
    assert {n for n in names if n[1] != "0"} == {(g, m, w) for g in ("16", "32", "64") for m in "123" for w in "234"}
    assert len([n for n in functions if re.match(r"_ZN12_GLOBAL__N_114vd_grid_kernelILb", n)]) == 2


@pytest.mark.parametrize("lanes", [16, 32, 64])
def test_conformations_on_the_device_are_read_without_exchanges(functions, lanes):
    """vd_eval_kernel on device memory: every lane loads its own numbers; only conformations in host
    memory come in one load and are handed round."""
    body = {host: next(b for n, b in functions.items() if n.startswith("_ZN12_GLOBAL__N_114vd_eval_kernelILi%dELb%dE" % (lanes, host)))
            for host in (0, 1)}
    assert not re.search(r"call [^@]*@_ZN3vdk\d+(gbcast|gget)", body[0])
    assert len(re.findall(r"call [^@]*@_ZN3vdk6gbcast", body[1])) == 7
