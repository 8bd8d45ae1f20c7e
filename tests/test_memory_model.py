"""The cross-workgroup hand-offs (grid reductions, flags, counters) of the
cooperative kernels publish with an agent-scope release: an L2 write-back
(buffer_wbl2) that must have completed before the flag or counter update a
reader on another XCD acquires.  hipcc for gfx950 drops that wait when the
source already waited on vmcnt before the release, so the kernels release
through rnpx::release_agent (fence + explicit wait).  This compiles the
kernel sources to gfx950 assembly (CPU only, with the library's flags) and
checks that every buffer_wbl2 is followed by s_waitcnt vmcnt(0) before the
next memory instruction.

Three hand-offs have no release: the outer-block kernel's grid-wide steps and the
triangular solves store their data through the caches (agent-scope relaxed stores,
sc1) and then a mark or flag, so each such mark must have an s_waitcnt vmcnt(0)
between it and the data before it (for the grid-wide steps in every wave: before the
workgroup barrier that precedes the mark); the real LU panel's words carry their
column's tag, so each must be one 8-byte access.  Checked per kernel in the same
assembly."""
import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rnp2_amd", "csrc")
SOURCES = ["rnpx_trsm.hip", "rnpx_cqr.hip", "rnpx_lu.hip", "rnpx_panel.hip", "rnpx_batched.hip"]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def unwaited_writebacks(asm):
    """Number of buffer_wbl2 not followed by s_waitcnt vmcnt(0) before the
    next vector-memory instruction, and the total."""
    total = bad = 0
    pending = False
    for line in asm.splitlines():
        s = line.strip()
        if s.startswith("buffer_wbl2"):
            total += 1
            pending = True
            continue
        if pending and s.startswith("s_waitcnt") and re.search(r"vmcnt\(0\)", s):
            pending = False
            continue
        if pending and re.match(r"(global_|buffer_|flat_|scratch_)", s):
            bad += 1
            pending = False
    return bad, total


def compile_asm(src, out_dir):
    out = os.path.join(out_dir, src + ".s")
    cmd = [HIPCC, "-x", "hip", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-O3", "-std=c++17",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"),
           os.path.join(CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return open(out).read()


@pytest.fixture(scope="module")
def asm():
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    with tempfile.TemporaryDirectory() as d:
        with cf.ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
            return dict(zip(SOURCES, ex.map(lambda s: compile_asm(s, d), SOURCES)))


def functions(asm):
    """name -> its lines, of every function in the assembly."""
    out, cur = {}, None
    for line in asm.splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            cur = out.setdefault(m.group(1), [])
        elif re.match(r"\.Lfunc_end", line):
            cur = None
        elif cur is not None:
            cur.append(line.split(";")[0].strip())
    return out


DATA = r"(global|flat)_store_(dwordx[24]|b64|b128)\b.*\bsc1"
WAIT = r"s_waitcnt\b.*vmcnt\(0\)"


def unwaited_marks(lines, mark, barrier):
    """Marks (stores matching `mark`) that a data store (sc1) may still be on its
    way behind, and the marks in all.  Walking back from the mark: the barrier
    first, where there is one, then s_waitcnt vmcnt(0) before any data store."""
    total = bad = 0
    for i, s in enumerate(lines):
        if not re.match(mark, s):
            continue
        total += 1
        seen_barrier, ok = not barrier, False
        for t in reversed(lines[:i]):
            if t.startswith("s_barrier"):
                if seen_barrier and barrier:
                    break
                seen_barrier = True
            elif re.match(WAIT, t):
                if seen_barrier:
                    ok = True
                    break
            elif re.match(DATA, t):
                break
        bad += not ok
    return bad, total


def test_marks_wait_for_written_through_data(asm):
    # grid-wide steps: one in blk_columnwise, two in the block kernel (reduce and
    # gather); a byte mark each
    cqr = {n: unwaited_marks(f, r"(global|flat)_store_byte\b.*sc1", True) for n, f in functions(asm["rnpx_cqr.hip"]).items()}
    for name, least in (("cqr_block_kernel", 2), ("blk_columnwise", 1)):
        got = [v for n, v in cqr.items() if name in n]
        assert len(got) == 1 and got[0][0] == 0 and got[0][1] >= least, (name, got)
    # triangular solves: the flag, a word, after x; one kernel per type and form
    trsm = {n: f for n, f in functions(asm["rnpx_trsm.hip"]).items() if "trsm_tri_kernel" in n}
    assert len(trsm) == 24
    for name, f in trsm.items():
        last = max(i for i, s in enumerate(f) if re.match(DATA, s))
        tail = f[last:]  # the abort flag's store, a word too, comes before x
        assert unwaited_marks(tail, r"global_store_dword\b.*sc1", False) == (0, 1), name


def test_lu_words_are_single_accesses(asm):
    f = next(f for n, f in functions(asm["rnpx_lu.hip"]).items() if "lu_row_panel_kernel" in n)
    stores = [s for s in f if re.match(r"(global|flat)_store\b|(global|flat)_store_\w+\b.*sc1", s)]
    words = [s for s in stores if "dwordx2" in s]
    # eight columns unrolled: a row's two words and a candidate's word each; the
    # abort flag (one dword) is the only other
    assert len(words) >= 3 * 8
    assert all(re.match(r"global_store_(dwordx2|dword)\b", s) for s in stores)
    loads = [s for s in f if re.match(r"global_load_\w+\b.*sc1", s)]
    assert sum("dwordx2" in s for s in loads) >= 5 * 8 and all(re.match(r"global_load_(dwordx2|dword)\b", s) for s in loads)


def test_an_unwaited_mark_is_seen():
    mark = r"global_store_byte\b.*sc1"
    data, wait, bar, byte = ("global_store_dwordx2 v[0:1], v[2:3], off sc1", "s_waitcnt vmcnt(0)", "s_barrier",
                             "global_store_byte v1, v0, s[4:5] sc1")
    assert unwaited_marks([data, wait, bar, byte], mark, True) == (0, 1)
    assert unwaited_marks([data, bar, wait, byte], mark, True) == (1, 1)  # other waves' data
    assert unwaited_marks([data, bar, byte], mark, True) == (1, 1)
    assert unwaited_marks([wait, data, bar, byte], mark, True) == (1, 1)
    assert unwaited_marks([data, byte], mark, False) == (1, 1)
    assert unwaited_marks([data, wait, byte], mark, False) == (0, 1)


def test_every_l2_writeback_is_waited_on(asm):
    report = {s: unwaited_writebacks(a) for s, a in asm.items()}
    print(report)
    assert sum(t for _, t in report.values()) > 0, "no release found: the check would pass vacuously"
    for src in ("rnpx_cqr.hip", "rnpx_lu.hip", "rnpx_panel.hip"):
        assert report[src][1] > 0, (src, report)
    assert all(b == 0 for b, _ in report.values()), report


def test_checker_flags_an_unwaited_writeback():
    bad_asm = "\tglobal_store_dwordx2 v1, v[2:3], s[4:5]\n\ts_waitcnt vmcnt(0)\n\tbuffer_wbl2 sc1\n" \
              "\tglobal_store_dword v0, v1, s[6:7] sc1\n"
    good_asm = "\tglobal_store_dwordx2 v1, v[2:3], s[4:5]\n\tbuffer_wbl2 sc1\n\ts_waitcnt vmcnt(0)\n" \
               "\tglobal_store_dword v0, v1, s[6:7] sc1\n"
    assert unwaited_writebacks(bad_asm) == (1, 1)
    assert unwaited_writebacks(good_asm) == (0, 1)
