"""The order in which workgroups take work items (attn_common.h: spread_workgroup and
work_position), compiled for the host and checked on the CPU: every item once, a whole
round's group on one XCD, each shader engine's share of every group, launches of fewer
than 8 groups starting with the longest query blocks of each; and fast_div."""
from __future__ import annotations

import shutil
import subprocess
from collections import Counter
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def dump_bin(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("wm") / "work_map_dump"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", f"-I{REPO / 'include'}",
                    f"-I{REPO / 'tilemix_amd' / 'csrc'}", str(REPO / "tests" / "native" / "work_map_dump.cpp"),
                    "-o", str(out)], check=True, capture_output=True)
    return out


def _run(dump_bin, *args):
    return subprocess.run([str(dump_bin), *map(str, args)], check=True, capture_output=True, text=True).stdout


def test_fast_div(dump_bin):
    assert int(_run(dump_bin, "--div")) == 0


@pytest.mark.parametrize("ilv", [1, 2, 3, 4])
@pytest.mark.parametrize("groups,m_blocks,group", [(64, 32, 3), (64, 15, 4), (4, 13, 7), (13, 5, 2), (9, 7, 1),
                                                   (7, 1, 1), (1, 1, 1), (24, 3, 5), (8, 2, 8), (3, 256, 7)])
def test_launch_order(dump_bin, groups, m_blocks, group, ilv):
    rows = [tuple(map(int, ln.split())) for ln in _run(dump_bin, groups, m_blocks, group, ilv).splitlines()]
    ipg = m_blocks * group
    done = [(g, i) for _, g, i in rows if g >= 0]
    assert sorted(done) == [(g, i) for g in range(groups) for i in range(ipg)]
    whole = groups // 8 * 8
    for bid, g, _ in rows:
        assert g < 0 or g >= whole or g % 8 == bid % 8
    per_xcd = len(rows) // 8
    if 32 < per_xcd <= 64:
        return  # every workgroup starts at once: test_two_workgroups_per_cu
    # the dispatcher deals an XCD's workgroups to four shader engines in turn: every engine gets
    # its share of every whole-round group (within the partial turns at the ends of a chunk)
    for x in range(8):
        share = Counter((g, (bid // 8) % 4) for bid, g, _ in rows if g >= 0 and g < whole and bid % 8 == x)
        for g in {g for g, _ in share}:
            counts = [share[g, e] for e in range(4)]
            assert max(counts) - min(counts) <= 2, (x, g, counts)
    # the groups past the whole rounds: ilv at a time, item by item, longest first
    tail = [(g - whole, i) for _, g, i in sorted(rows, key=lambda r: r[0]) if g >= whole]
    for c in range(0, groups - whole, ilv):
        chunk = [i for g, i in tail if c <= g < c + ilv]
        kc = min(ilv, groups - whole - c)
        # rotations move a position by less than one turn of the four engines on 8 XCDs
        assert all(abs(i - w // kc) <= 32 // kc + 1 for w, i in enumerate(chunk))


@pytest.mark.parametrize("groups,m_blocks,group", [(8, 11, 3), (8, 16, 3), (8, 16, 4), (16, 8, 3), (8, 33, 1)])
def test_two_workgroups_per_cu(dump_bin, groups, m_blocks, group):
    """33 to 64 workgroups per XCD, item 0 the longest query block: workgroup j + 32 shares the CU
    of workgroup j.  The longest items are alone; of the others, longest goes with shortest."""
    rows = [tuple(map(int, ln.split())) for ln in _run(dump_bin, groups, m_blocks, group, 4).splitlines()]
    n = len(rows) // 8
    assert 32 < n <= 64
    for x in range(8):
        rank = sorted(range(n), key=lambda j: (rows[8 * j + x][2], rows[8 * j + x][1]))  # positions, longest first
        at = {j: r for r, j in enumerate(rank)}
        alone = [at[j] for j in range(n - 32, 32)]
        assert alone == list(range(64 - n))
        assert all(at[j] + at[j + 32] == 63 for j in range(n - 32))


@pytest.mark.parametrize("groups,m_blocks,group", [(8, 65, 1), (8, 24, 4), (8, 18, 4), (16, 15, 3), (8, 13, 5)])
def test_three_workgroups_per_cu(dump_bin, groups, m_blocks, group):
    """65 to 96 workgroups per XCD of which a CU holds three: every item once, and workgroup j + 32,
    on the CU of workgroup j, is the shorter the longer that is; the rest stays longest first."""
    rows = [tuple(map(int, ln.split())) for ln in _run(dump_bin, groups, m_blocks, group, 4, 3).splitlines()]
    n = len(rows) // 8
    assert 64 < n <= 96
    assert sorted((g, i) for _, g, i in rows) == [(g, i) for g in range(groups) for i in range(m_blocks * group)]
    for x in range(8):
        rank = sorted(range(n), key=lambda j: (rows[8 * j + x][2], rows[8 * j + x][1]))
        at = {j: r for r, j in enumerate(rank)}
        assert all(at[j] == j for j in range(32))
        assert all(at[j + 32] == 63 - j for j in range(32))
        assert all(at[j] == j for j in range(64, n))


@pytest.mark.parametrize("per_cu", [2, 3])
@pytest.mark.parametrize("groups,m_blocks,group", [(4, 16, 7), (1, 33, 8), (7, 13, 4), (4, 22, 7), (5, 31, 4), (1, 96, 8),
                                                   (2, 65, 4)])
def test_shared_cus_with_fewer_than_8_groups(dump_bin, groups, m_blocks, group, per_cu):
    """33 to 96 workgroups per XCD of launches whose groups are dealt over all XCDs: every item once; with
    two per CU and the groups interleaved all at once, the longest items are alone."""
    rows = [tuple(map(int, ln.split())) for ln in _run(dump_bin, groups, m_blocks, group, 4, per_cu).splitlines()]
    n = len(rows) // 8
    assert 32 < n <= 96
    assert sorted((g, i) for _, g, i in rows if g >= 0) == [(g, i) for g in range(groups)
                                                            for i in range(m_blocks * group)]
    if n <= 64 and groups <= 4:
        for x in range(8):
            item = [rows[8 * j + x][2] for j in range(n)]
            alone = [item[j] for j in range(n - 32, 32) if item[j] >= 0]
            paired = [item[j] for j in (*range(n - 32), *range(32, n)) if item[j] >= 0]
            assert not alone or max(alone) <= min(paired)


@pytest.mark.parametrize("per_cu", [2, 3])
@pytest.mark.parametrize("groups,m_blocks,group", [(8, 11, 3), (8, 24, 4), (4, 16, 7), (64, 15, 4), (3, 40, 1)])
def test_without_the_causal_limit(dump_bin, groups, m_blocks, group, per_cu):
    """Items of equal length: the rotated order, whatever number of workgroups a CU holds, and
    launches of fewer than 8 groups take them one after the other (within a turn of the rotation)."""
    rows = _run(dump_bin, groups, m_blocks, group, 4, per_cu, 0)
    ilv = 4 if groups >= 8 else 1
    assert rows == _run(dump_bin, groups, m_blocks, group, ilv, 1, 1)  # one workgroup per CU: nothing shared
    if groups < 8:
        order = [g for g, _ in (tuple(map(int, ln.split()[1:])) for ln in rows.splitlines()) if g >= 0]
        assert all(abs(g - w // (m_blocks * group)) <= (w % (m_blocks * group) < 32 or
                                                        w % (m_blocks * group) >= m_blocks * group - 32)
                   for w, g in enumerate(order))
    done = [tuple(map(int, ln.split()[1:])) for ln in rows.splitlines()]
    assert sorted(p for p in done if p[0] >= 0) == [(g, i) for g in range(groups) for i in range(m_blocks * group)]
