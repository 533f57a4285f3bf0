"""What the GEMM kernels' gfx950 assembly has to look like, read from a compile of gemm.hip with the library's flags (no GPU): where a
matrix instruction is an asm statement, or a wait stands between two stores, the sources alone do not show it."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutlass-kernels_amd", "csrc")
FLAGS = ["-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument", "-fno-gpu-rdc", "--offload-device-only"]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> its instructions, in the order of the text"""
    out = str(tmp_path_factory.mktemp("asm") / "gemm.s")
    subprocess.run(["/opt/rocm/bin/hipcc"] + FLAGS + ["-S", "-o", out, "gemm.hip"], cwd=CSRC, check=True, capture_output=True)
    found = {}
    for m in re.finditer(r"^(_ZN3cfk12_GLOBAL__N_1\d+(gemm_kernel\w*?)I(\S*?)EEv\S*):.*?\n(.*?)\.Lfunc_end", open(out).read(), re.S | re.M):
        name = m.group(2) + "<" + ",".join(re.findall(r"L[bi](\d+)", m.group(3))) + ">"
        lines = [x.strip() for x in m.group(4).splitlines()]
        found[name] = [x for x in lines if x and x[0] not in ";."]
    return found


def _through(ins):
    return [i for i, x in enumerate(ins) if x.startswith("global_store_dwordx4") and x.endswith("sc1")]


def _waits(ins):
    """(index, n) of every wait for all but n vector memory instructions"""
    return [(i, int(m.group(1))) for i, x in enumerate(ins) if (m := re.search(r"s_waitcnt.*vmcnt\((\d+)\)", x))]


@pytest.mark.parametrize("name", ["gemm_kernel16_tile_c<%d,%s>" % (nn, t) for nn in (0, 1) for t in ("256,128", "128,128", "128,64")] +
                         ["gemm_kernel_f32_c<128>", "gemm_kernel_f32_c<64>"])
def test_tiles_over_c_do_not_wait_for_their_stores(kernels, name):
    ins = kernels[name]
    st = _through(ins)
    assert len(st) >= 2
    # all of C is asked for in front of the first store, so the last piece of it lies behind none of them
    assert min([n for i, n in _waits(ins) if st[0] < i < st[-1]], default=len(st)) >= len(st) - 1, name


@pytest.mark.parametrize("name", ["gemm_kernel16_tile<%d,%s>" % (nn, t) for nn in (0, 1) for t in ("256,128", "128,128", "128,64")] +
                         ["gemm_kernel_f32<128>", "gemm_kernel_f32<64>"])
def test_tiles_without_c_carry_no_code_for_it(kernels, name):
    # (calls with C take the kernels above)
    ins = kernels[name]
    st = _through(ins)
    assert len(st) >= 2 and not [x for x in ins if x.startswith("global_load_dwordx4")], name
    assert not [i for i, _ in _waits(ins) if st[0] < i < st[-1]], name


BLOCK_KERNELS = [("gemm_kernel16%s" % (k % nn), rows // 16 // 2, cols) for nn in (0, 1)
                 for k, rows, cols in (("<%d,4>", 256, 256), ("<%d,3>", 256, 192), ("_rows<%d,6,4>", 192, 256), ("_rows<%d,6,3>", 192, 192),
                                       ("_rows<%d,10,4>", 320, 256))]


@pytest.mark.parametrize("name", [k[0] for k in BLOCK_KERNELS])
def test_nothing_touches_the_accumulators_between_the_asm_multiplies(kernels, name):
    # the multiplies of these kernels are asm statements, whose latency the compiler does not see: a copy or a spill of an
    # accumulator between them, or of an operand right in front of one, would read or write it too early
    ins = kernels[name]
    at = [i for i, x in enumerate(ins) if x.startswith("v_mfma")]
    other = {x.split()[0] for x in ins[at[0]:at[-1] + 1] if not x.startswith(("v_mfma", "s_", "ds_", "buffer_load_dwordx4"))}
    assert other <= {"v_add_u32_e32", "v_add3_u32"}, (name, other)   # LDS and scalar-offset addresses


@pytest.mark.parametrize("name,blocks,cols", BLOCK_KERNELS)
def test_blocks_without_c_wait_for_nothing_between_their_stores(kernels, name, blocks, cols):
    ins = kernels[name]
    waits = {i for i, _ in _waits(ins)}
    run = longest = 0
    for i, x in enumerate(ins):
        if i in waits: run = 0
        elif x.startswith("global_store_dwordx4") and x.endswith("sc1"): run += 1
        longest = max(longest, run)
    assert longest >= blocks * 2, (name, longest)   # two stores for each row of blocks of a wave


@pytest.mark.parametrize("name,blocks", [k[:2] for k in BLOCK_KERNELS if k[1] <= 8])
def test_blocks_over_c_ask_for_all_of_it_before_their_first_store(kernels, name, blocks):
    # two forms (through the caches and past them), two pieces for each row of blocks of a wave, none of them asked for behind a wait for
    # the others or behind a store: the compiler likes to move the first one into the branch around its store
    ins = kernels[name]
    start = [i for i, x in enumerate(ins) if x.startswith("v_mfma")][-1]
    waits = {i for i, n in _waits(ins) if n == 0}
    runs, run, waited = [], 0, False
    for i in range(start, len(ins)):
        if i in waits: waited = run > 0
        elif ins[i].startswith("global_load_dwordx4"):
            assert not waited, (name, i - start)
            run += 1
        elif ins[i].startswith("global_store") and run: runs, run, waited = runs + [run], 0, False
    assert runs == [2 * blocks] * 2, (name, runs)
