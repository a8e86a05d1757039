"""What the compiler makes of the expert GEMMs (ggemm.hip): properties of the generated code that the kernels' speed or
their waits rest on and that no result shows."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "optimus-lm_amd", "csrc")
# template arguments of ggemm_kernel, in order
FIELDS = ("BM", "AKIND", "BKIND", "EPI", "GATHER", "ROWW", "ACCUM", "EDGE", "ONCE", "DENSE")
EPI_WGRAD = 3


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """[(template arguments, assembly lines, notes)] of the library's build."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    import build as library_build
    out = str(tmp_path_factory.mktemp("asm") / "ggemm.s")
    flags = [f for f in library_build.HIPCC_FLAGS if f != "-shared"]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(CSRC, "ggemm.hip"), "-o", out], check=True,
                   capture_output=True)
    text = open(out).read()
    notes = {m.group(1): dict(re.findall(r"\.(\w+_spill_count):\s*(\d+)", m.group(0)))
             for m in re.finditer(r"\.name:\s+(\S+).*?\.wavefront_size", text, re.S)}
    found = []
    for name in sorted(set(re.findall(r"^(\S*ggemm_kernel\S+):", text, re.M))):
        arguments = dict(zip(FIELDS, map(int, re.findall(r"L[ib](\d+)E", name))))
        assert len(arguments) == len(FIELDS)
        start = text.index("\n" + name + ":")
        found.append((arguments, text[start:text.index(".Lfunc_end", start)].split("\n"), notes[name]))
    assert len(found) > 30
    return found


def test_step_1_is_loaded_ahead_only_where_the_stores_are_counted(kernels):
    """Loads of a tile's step 1 in front of the last one's stores are of use where the first wait leaves the stores out;
    anywhere else they are code, and a wait for what is behind them.  128x128 row products: as many direct loads in every kernel."""
    counts = set()
    for k, lines, _ in kernels:
        ahead = any("s_waitcnt vmcnt(16) lgkmcnt(0)" in line for line in lines)
        assert ahead == (k["EPI"] == EPI_WGRAD and not k["EDGE"]), k
        if k["BM"] == 128 and k["EPI"] != EPI_WGRAD:
            counts.add(sum("global_load_lds_dwordx4" in line and not line.endswith(" nt") for line in lines))
    assert len(counts) == 1


def test_first_steps_of_128x128_tiles_are_loaded_ahead_of_the_first_wait(kernels):
    """All eight loads that step 1 of a tile needs are under way when a wavefront first waits, for step 0."""
    for k, lines, _ in kernels:
        if k["BM"] == 128:
            first = [line.split()[1] for line in lines if re.match(r"\s*s_waitcnt vmcnt\(\d+\) lgkmcnt\(0\)$", line)]
            assert set(first) == {"vmcnt(8)", "vmcnt(0)"}, k


def test_128x128_row_products_have_each_step_once(kernels):
    """Even and odd steps, of tiles with both row units and of tiles with one: 32 MFMAs a step or 16.  Short launches fetch
    their code cold."""
    for k, lines, _ in kernels:
        if k["BM"] == 128 and k["EPI"] != EPI_WGRAD:
            assert sum("v_mfma_f32_16x16x32_bf16" in line for line in lines) == 2 * (32 + 16), k


def test_weight_gradients_start_a_tile_with_stores_under_way(kernels):
    """From the wait that leaves the last tile's 16 stores out to the first MFMA nothing else waits for memory: what the compiler
    believes to be still on its way there it would wait for together with the stores."""
    seen = 0
    for k, lines, _ in kernels:
        if k["BM"] == 256 and k["EPI"] == EPI_WGRAD:
            at = next(i for i, line in enumerate(lines) if "s_waitcnt vmcnt(16) lgkmcnt(0)" in line)
            until = next(i for i in range(at, len(lines)) if "v_mfma" in lines[i])
            assert not any("vmcnt(" in line or "scratch_" in line for line in lines[at + 1:until]), k
            seen += 1
    assert seen == 8


def test_no_vector_register_is_spilled(kernels):
    """Nor more than a few scalar ones, into lanes of a vector register (a dense expert's operands stand beside the others')."""
    for k, lines, notes in kernels:
        assert int(notes["vgpr_spill_count"]) == 0 and int(notes["sgpr_spill_count"]) <= (16 if k["DENSE"] else 4), k
        assert not any("scratch_" in line for line in lines), k


def test_counted_stores_stay_behind_the_loads_they_follow(kernels):
    """The first wait of a tile leaves the 16 youngest operations out, which are the last tile's stores only while none of them
    stands ahead of the direct loads."""
    for k, lines, _ in kernels:
        if k["BM"] == 256 and k["EPI"] == EPI_WGRAD:
            at = [i for i, line in enumerate(lines) if "stores from here on" in line]
            assert len(at) == 1, k
            stores = [i for i, line in enumerate(lines) if re.match(r"\s*(global|buffer)_store_dwordx4", line)]
            assert len(stores) >= 32 and min(stores) > at[0], k       # past the caches and through them
            assert max(i for i, line in enumerate(lines) if "global_load_lds" in line) < at[0], k


def test_row_products_read_their_arguments_when_they_start(kernels):
    """A few wide reads in all, and none from the first tile on: each is a trip through the scalar cache that a block waits for."""
    for k, lines, _ in kernels:
        if k["EPI"] != EPI_WGRAD:
            reads = [i for i, line in enumerate(lines) if re.match(r"\s*s_load_dword", line)]
            assert len(reads) <= (16 if k["DENSE"] else 11), (k, len(reads))
            assert max(reads) < min(i for i, line in enumerate(lines) if "v_mfma" in line), k
