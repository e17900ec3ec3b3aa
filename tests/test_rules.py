"""The rules that choose kernels and store policies (dg_rules.hpp, host build) on both sides of their
lines, at the sizes where the two sides were measured; and that a store policy is still there after
the compiler."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "rules_host")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "host", "rules_host.cpp")], check=True)

    def ask(*words):
        line = " ".join(str(int(w) if isinstance(w, bool) else w) for w in words)
        return int(subprocess.run([exe], input=line, capture_output=True, text=True, check=True).stdout)

    return ask


# dim, p, FP64, line kernel, curved, state in MB; faster cached
STORE = [(3, 3, True, True, False, 8.6, False), (3, 3, True, True, False, 84, True), (3, 3, False, True, False, 119, True),
         (2, 1, False, True, False, 3.2, False), (2, 2, False, False, False, 7.1, True), (2, 1, True, True, False, 320, True),
         (3, 3, False, False, False, 20, False), (3, 6, True, False, False, 24, True), (3, 2, False, False, False, 84, True),
         (3, 6, True, False, False, 127, False), (2, 3, False, False, False, 134, False), (2, 1, False, False, False, 134, True),
         (3, 3, True, True, True, 62, True), (3, 3, True, True, True, 84, False), (3, 1, True, True, True, 170, True),
         (3, 4, False, False, True, 122, False)]


@pytest.mark.parametrize("dim,p,fp64,line,curved,mb,cached", STORE)
def test_store_policy(rules, dim, p, fp64, line, curved, mb, cached):
    assert rules("store", dim, p + 1, fp64, line, curved, mb) == cached


EC, GEN, CONS = 0, 1, 2
# dim, p, FP64, form, cells a side; faster in small blocks
SMALL = [(3, 3, True, EC, 10, True), (3, 3, True, EC, 11, False), (2, 5, True, EC, 41, True), (3, 6, True, EC, 2, False),
         (3, 3, False, EC, 10, True), (3, 3, False, EC, 12, False), (3, 4, False, EC, 8, True), (3, 4, False, EC, 9, False),
         (3, 6, False, EC, 6, True), (3, 6, False, EC, 7, False), (2, 5, True, GEN, 29, True), (2, 3, True, GEN, 27, False),
         (3, 1, True, CONS, 16, True), (3, 1, True, CONS, 18, False), (3, 2, True, CONS, 11, True),
         (3, 2, True, CONS, 12, False), (2, 3, True, CONS, 14, False), (2, 4, True, CONS, 50, True),
         (2, 1, True, CONS, 106, True)]


@pytest.mark.parametrize("dim,p,fp64,form,n,small", SMALL)
def test_small_meshes_block(rules, dim, p, fp64, form, n, small):
    assert rules("small", dim, p + 1, fp64, form, n ** dim) == small


# dim, p, boundary faces, stage of a step, cells a side; faster in the line kernel
CONSERVATIVE = [(3, 3, False, False, 12, False), (3, 3, False, True, 12, True), (3, 3, False, False, 15, True),
                (3, 5, False, False, 8, False), (3, 5, False, True, 7, True), (3, 5, False, False, 10, True),
                (3, 2, False, False, 13, False), (3, 2, False, False, 15, True), (3, 1, False, False, 23, False),
                (3, 1, False, True, 23, True), (3, 1, False, True, 20, False), (3, 1, False, False, 30, True),
                (3, 6, False, False, 14, False), (2, 4, False, True, 300, False), (3, 3, True, False, 7, True),
                (3, 1, True, False, 18, False), (3, 1, True, False, 23, True)]


@pytest.mark.parametrize("dim,p,boundary,stage,n,line", CONSERVATIVE)
def test_conservative_line_kernel(rules, dim, p, boundary, stage, n, line):
    assert rules("conservative", dim, p + 1, boundary, stage, n ** dim) == line


@pytest.mark.parametrize("dim,p,fp64,blocks,small", [
    (2, 4, True, 250, True), (2, 4, True, 350, False), (3, 3, True, 256, True), (3, 2, True, 125, True),
    (3, 2, True, 182, False), (3, 4, True, 182, False), (3, 1, True, 253, False), (3, 1, False, 188, True),
    (3, 2, False, 250, False), (3, 6, True, 256, True)])
def test_batch_small_tile(rules, dim, p, fp64, blocks, small):
    assert rules("batch", dim, p + 1, fp64, blocks) == small


@pytest.mark.parametrize("dim,p,fp64,early", [(2, 1, False, False), (2, 2, False, False), (2, 3, False, True),
                                              (3, 1, False, True), (2, 1, True, True)])
def test_butcher_prefetch(rules, dim, p, fp64, early):
    assert rules("prefetch", dim, p + 1, fp64) == early


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_both_store_policies_are_in_the_code(tmp_path):
    """The state's four stores once streamed and once not, beside S2's four streamed ones."""
    out = str(tmp_path / "s.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=on", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", out,
                    os.path.join(HERE, "host", "stage_store.hip")], check=True, capture_output=True)
    stores = [x for x in open(out).read().splitlines() if re.search(r"\bglobal_store_dwordx2\b", x)]
    assert sum(" nt" in x for x in stores) == 8 and sum(" nt" not in x for x in stores) == 4
