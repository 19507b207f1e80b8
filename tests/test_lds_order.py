"""CPU: the decoders that pass bytes between a wave's lanes through LDS (the
wave kernels' wave_decode, k_gemv_gulp's tier-2 exchange) order them by a
wavefront fence, which the optimiser must honour. A wave barrier alone is no
memory operation to it, and the exchanges are written and read in different
types, which it may take for disjoint memory. Read in the compiler's IR before
any pass has run."""

import os
import re
import shutil
import subprocess

import pytest

from drinkme_amd import build

HIPCC = "/opt/rocm/bin/hipcc"
# fences a block's decode takes by profile (0 sip, 1 balanced, 2 gulp): after the tail words, after each
# resolved tier's bytes, and before the words are written again
FENCES = {0: 2, 1: 3, 2: 4}
# and wave_wide's: in the writer of a level's bytes, and after each read of them
WIDE = {0: 0, 1: 2, 2: 3}


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("ir") / "kernels.ll")
    subprocess.run([build._hipcc(), *build.device_flags(), "--cuda-device-only", "-S", "-emit-llvm", "-Xclang",
                    "-disable-llvm-passes", os.path.join(build.CSRC, "kernels.hip"), "-o", out], check=True,
                   capture_output=True)
    bodies, name = {}, None
    with open(out) as f:
        for line in f:
            m = re.match(r"define .*?@(\w+)\(", line)
            if m:
                name = m.group(1)
                bodies[name] = []
            elif line.startswith("}"):
                name = None
            elif name is not None:
                bodies[name].append(line)
    return bodies


def _syncs(functions, body):
    """The fences of a body, calls of a function of its own that fences and
    barriers counted; and the wave barriers no fence stands in front of."""
    fence = re.compile(r'fence syncscope\("wavefront"\) acq_rel')
    barrier = re.compile(r"call void @llvm\.amdgcn\.wave\.barrier\(")
    count = bare = 0
    fenced = False
    for line in body:
        callee = re.search(r"call .*?@(\w+)\(\)", line)
        inner = functions.get(callee.group(1)) if callee else None
        for at in inner if inner is not None else [line]:
            if fence.search(at):
                count, fenced = count + 1, True
            elif barrier.search(at):
                bare, fenced = bare + (not fenced), False
    return count, bare


def test_every_exchange_is_fenced(functions):
    decoders, gulp, wide = 0, {}, {}
    for name, body in functions.items():
        decode = re.match(r"_ZN12_GLOBAL__N_111wave_decodeILi(\d)ELi\dEEEv", name)
        kernel = re.match(r"_ZZ?N12_GLOBAL__N_1(11k_gemv_gulpI\w*?EEEv)", name)  # (with its lambdas)
        if decode:
            decoders += 1
            assert _syncs(functions, body) == (FENCES[int(decode.group(1))], 0), name
        elif kernel:
            count, bare = _syncs(functions, body)
            assert bare == 0, name
            gulp[kernel.group(1)] = gulp.get(kernel.group(1), 0) + count
        through = re.match(r"_ZZ?N12_GLOBAL__N_19wave_wideILi(\d)EEEv", name)  # (with its lambdas)
        if through:
            count, bare = _syncs(functions, body)
            assert bare == 0, name
            wide[int(through.group(1))] = wide.get(int(through.group(1)), 0) + count
    assert decoders == 6
    assert wide == WIDE, wide
    # around the read of the tier-2 bytes
    assert gulp and set(gulp.values()) == {2}, gulp
