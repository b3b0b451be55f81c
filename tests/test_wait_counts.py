"""Static check of the hand-written wait counts in the MFMA kernels' machine code.

The tiled and the mid-M kernel stream their activation tiles global -> LDS with LDS-direct loads and wait for a tile
with an inline `s_waitcnt vmcnt(N)`, N > 0: vector-memory operations complete in order, so "at most N outstanding"
means the tile has landed only if the wave has issued at least N vector-memory instructions behind the tile's last
LDS-direct load.  N is written by hand next to the loads it counts (gptq4_gemm.hip, gptq4_kslice.hip); a compiler that
merged, dropped or hoisted one of those loads above the LDS-direct loads would make the wait return early and the MFMAs
read a tile that is still in flight - with results that are wrong only sometimes.  This test compiles the two files to
gfx950 assembly and follows every path of every kernel variant from the kernel's entry on, with the tiles requested on it
(groups of LDS-direct loads) and the vector-memory instructions behind each.  A loop is entered with two tiles requested: the
first such wait on a path is for the older one, every later wait for all that have been requested by then, and a tile's count
must reach the N of the wait it is for (or of an earlier one).
"""
import importlib.util
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "gptq-triton_amd" / "csrc"

VMEM = re.compile(r"^(buffer|global|flat|scratch)_(load|store|atomic)")
WAIT = re.compile(r"^s_waitcnt\b.*\bvmcnt\((\d+)\)")
LABEL = re.compile(r"^(\.LBB\d+_\d+):")
BRANCH = re.compile(r"^(s_c?branch\w*)\s+(\.LBB\d+_\d+)")


def _build_flags():
    spec = importlib.util.spec_from_file_location("_gptq4_build", ROOT / "gptq-triton_amd" / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod._hipcc(), [f for f in mod.HIPCC_FLAGS if f != "-fPIC"]


def _assembly(source: Path, tmp: Path) -> str:
    hipcc, flags = _build_flags()
    out = tmp / (source.stem + ".s")
    res = subprocess.run([hipcc, *flags, "-w", "-S", "--cuda-device-only", str(source), "-o", str(out)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    return out.read_text()


def _kernels(asm: str):
    """(name, [(line, inline)]) per kernel function: instruction and label lines without comments; inline = the line
    stands between the markers the compiler puts around an asm statement of the source."""
    for m in re.finditer(r"^(_Z\w*gptq4_\w+_kernel\w*):.*$", asm, re.M):
        end = asm.index(".Lfunc_end", m.end())
        lines, inline = [], False
        for raw in asm[m.end():end].splitlines():
            if "#ASMSTART" in raw:
                inline = True
            elif "#ASMEND" in raw:
                inline = False
            line = raw.split(";")[0].strip()
            if line:
                lines.append((line, inline))
        yield m.group(1), lines


def _table_loads(text):
    """Indices of the LDS-direct loads of the rotary tables (waited for with vmcnt(0), behind the loop): in the order they are
    written, runs of them go through two buffers in turn, with no scalar offset."""
    tables, run = set(), []
    for i, l in enumerate(text + ["buffer_load_dword v0, v0, s[0:3], 0"]):
        if not VMEM.match(l):
            continue
        if l.split()[-1] == "lds":
            run.append(i)
            continue
        args = [[a.strip() for a in text[r].split(",")] for r in run]
        if len({a[1] for a in args}) > 1 and all(a[2].split()[0] == "0" for a in args):
            tables.update(run)
        run = []
    return tables


def _paths_to_waits(lines):
    """[(N, vector-memory instructions behind a tile's LDS-direct loads, index of the wait)] over all paths from the entry, for
    every hand-written wait and every tile it is for."""
    text = [l for l, _ in lines]
    label_at = {m.group(1): i for i, l in enumerate(text) if (m := LABEL.match(l))}
    waits = {i: int(m.group(1)) for i, l in enumerate(text) if (m := WAIT.match(l))}
    hand = {i: n for i, n in waits.items() if lines[i][1] and n > 0}
    if not hand:
        return []
    cap = max(hand.values()) + 1  # (counts beyond any wait's N are all the same)
    tables = _table_loads(text)
    results, seen = [], set()
    # state: (index, counts behind the tiles requested and not yet known to have landed, inside a tile's loads, a wait has passed)
    stack = [(0, (), False, False)]
    while stack:
        i, behind, inside, later = stack.pop()
        while i < len(text):
            if (i, behind, inside, later) in seen:
                break
            seen.add((i, behind, inside, later))
            cur = text[i]
            if waits.get(i) == 0:  # everything has landed (of the source's own: a loop ends here, and another one may follow)
                behind, inside, later = (), False, later and not lines[i][1]
            elif i in hand and behind:
                n = hand[i]
                for count in behind if later else behind[:1]:
                    results.append((n, count, i))
                behind, inside, later = () if later else tuple(c for c in behind[1:] if c < n), False, True
            if VMEM.match(cur):
                if cur.split()[-1] == "lds" and i not in tables:
                    if not inside:
                        behind, inside = behind + (0,), True
                    behind = tuple(min(c + 1, cap) for c in behind[:-1]) + (0,)
                else:
                    behind, inside = tuple(min(c + 1, cap) for c in behind), False
            if cur.startswith(("s_endpgm", "s_setpc")):
                break
            b = BRANCH.match(cur)
            if b:
                stack.append((label_at[b.group(2)], behind, inside, later))
                if b.group(1) == "s_branch":
                    break
            i += 1
    return sorted(set(results))


@pytest.fixture(scope="module")
def assemblies(tmp_path_factory):
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("hipcc not available")
    tmp = tmp_path_factory.mktemp("isa")
    return {name: _assembly(CSRC / name, tmp) for name in ("gptq4_gemm.hip", "gptq4_kslice.hip")}


ACT_ORDER_GEMM = re.compile(r"gptq4_gemm_kernelILi\dELi\dELb1E")  # <EPI, MT, PERM = true, ..>


@pytest.mark.parametrize("source,variants", [("gptq4_gemm.hip", 15), ("gptq4_kslice.hip", 48)])
def test_hand_written_wait_counts_match_the_loads_behind_the_lds_direct_loads(assemblies, source, variants):
    with_waits = 0
    for name, lines in _kernels(assemblies[source]):
        found = _paths_to_waits(lines)
        for n, behind, at in found:
            assert behind >= n, (f"{name}: a path reaches `{lines[at][0]}` with only {behind} vector-memory instructions "
                                 f"behind the activation tile's LDS-direct loads: the tile may not have landed")
        # (the act-order variants of the tiled kernel stage their tiles through registers and have no such wait)
        assert bool(found) != bool(ACT_ORDER_GEMM.search(name)), f"{name}: the scan sees {len(found)} paths to such a wait"
        with_waits += bool(found)
    assert with_waits == variants, f"{with_waits} kernel variants of {source} show such waits"


def test_the_scan_covers_the_96_row_tiles(assemblies):
    """Five variants (plain, wide strips, gate/up, whole and paired rotary heads) on both weight layouts."""
    tall = {name for name, lines in _kernels(assemblies["gptq4_kslice.hip"]) if re.search(r"kslice_kernelILi\dELi3E", name) and _paths_to_waits(lines)}
    assert len(tall) == 10


def test_the_scan_sees_a_missing_load():
    """The checker itself: a tile requested before the loop and at the top of every pass, the wait at the top."""
    def prog(loads_in_loop):
        body = [("buffer_load_dwordx4 v1, s[0:3], s4 offen lds", False)] + [("global_load_dword v9, v[4:5], off", False)] * 5
        body += [(".LBB0_1:", False), ("s_waitcnt vmcnt(4) lgkmcnt(0)", True), ("s_barrier", True),
                 ("buffer_load_dwordx4 v1, s[0:3], s4 offen lds", False), ("buffer_load_dwordx4 v2, s[0:3], s4 offen lds", False)]
        body += [("global_load_dword v6, v[4:5], off", False)] * loads_in_loop
        body += [("v_mfma_f32_32x32x16_f16 a[0:15], v[0:3], v[4:7], a[0:15]", False), ("s_cbranch_scc1 .LBB0_1", False), ("s_endpgm", False)]
        return body
    assert sorted(_paths_to_waits(prog(4))) == [(4, 4, 7), (4, 5, 7)]
    assert sorted(_paths_to_waits(prog(3))) == [(4, 3, 7), (4, 5, 7)]
    # a wait of the compiler's own (not between the asm markers) is not a checkpoint
    assert _paths_to_waits([(l, False) for l, _ in prog(3)]) == []


def test_the_scan_sees_a_missing_load_behind_the_second_tile_of_a_prologue():
    """Two tiles requested before the loop, the next one behind the wait in the loop: the first wait in the loop is for the second."""
    tile = [("buffer_load_dwordx4 v1, s[0:3], s4 offen lds", False)] * 2
    words = lambda n: [("buffer_load_dwordx2 v[6:7], v8, s[8:11], s5 offen", False)] * n

    def prog(behind_first, behind_second, in_loop):
        return (tile + words(behind_first) + tile + words(behind_second) + [("s_waitcnt vmcnt(9)", True), (".LBB0_1:", False)] + words(in_loop - 1) +
                [("s_waitcnt vmcnt(4) lgkmcnt(0)", True)] + tile + words(1) + [("s_cbranch_scc1 .LBB0_1", False), ("s_endpgm", False)])

    def short(*counts):
        return sorted({(n, behind) for n, behind, _ in _paths_to_waits(prog(*counts)) if behind < n})

    assert short(5, 2, 4) == []
    assert short(5, 0, 4) == [(4, 3), (9, 7)]  # the second tile's words requested in front of its rows
    assert short(4, 2, 4) == [(9, 8)]
    assert short(5, 2, 3) == [(4, 3)]
    # a tile that an earlier wait has covered needs no other
    assert short(5, 9, 2) == [(4, 2)] and (4, 10, 21) not in _paths_to_waits(prog(5, 9, 2))


def test_table_loads_are_told_from_a_tiles():
    """The rotary tables' loads behind the second tile are landed by the end of the loop only."""
    tables = [("buffer_load_dwordx4 v1, s[12:15], 0 offen lds", False), ("buffer_load_dwordx4 v1, s[16:19], 0 offen lds", False)] * 2
    tile = [("buffer_load_dwordx4 v1, s[0:3], 0 offen lds", False)] * 2
    word = [("buffer_load_dwordx2 v[6:7], v8, s[8:11], s5 offen", False)]
    body = tile + word * 3 + tables + [("s_waitcnt vmcnt(7)", True), ("s_waitcnt vmcnt(5)", True), ("s_waitcnt vmcnt(0)", True), ("s_endpgm", False)]
    assert [r[:2] for r in _paths_to_waits(body)] == [(7, 7)]
