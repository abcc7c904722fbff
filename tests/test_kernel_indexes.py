"""Index rules that kernels share with the host, checked over every lane on
the CPU: the headers hold plain constexpr functions, compiled here by the host
compiler alone. A wrong row would be an access outside the kernel's LDS, which
no result shows while the word it hits is unused.
"""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "metal-gauss_amd" / "csrc"


def _run(tmp_path, header: str, body: str, edit=None):
    """Compile `body` in a main() over `header` (its text replaced as `edit`
    says) and return its output as rows of ints."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    text = (CSRC / header).read_text()
    if edit is not None:
        assert text.count(edit[0]) == 1, edit[0]
        text = text.replace(*edit)
    (tmp_path / header).write_text(text)
    src = tmp_path / "main.cpp"
    src.write_text(f'#include <cstdint>\n#include <cstdio>\n#include "{header}"\n'
                   f"using namespace mg;\nint main() {{\n{body}\nreturn 0;\n}}\n")
    exe = tmp_path / "main"
    p = subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(p.stderr)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=60).stdout
    return [[int(x) for x in line.split()] for line in out.splitlines()]


# Which value's sum lane row r of reduce10_to_rows's q-th result holds, None
# for a sum of zeros.
ROW_VALUES = ((0, 2, 1, 3), (4, 6, 5, 7), (8, None, 9, None))


@pytest.mark.parametrize("abs_grad", [False, True])
def test_raster_backward_deposits_stay_in_their_rows(tmp_path, abs_grad):
    """Every lane that adds to the per-entry sums has a row of its own value,
    and the lanes that carry zeros (value 9 among them without |d uv|) add to
    one that exists."""
    flag = str(abs_grad).lower()
    rows = _run(tmp_path, "raster_slots.h", f"""
        std::printf("%d\\n", grad_rows({flag}));
        for (int q = 0; q < 3; ++q)
            for (int r = 0; r < 4; ++r) std::printf("%d %d %d\\n", q, r, deposit_row(q, r, {flag}));
        for (int l = 0; l < 64; ++l) std::printf("%d\\n", reduce18_slot(l));""")
    n = rows[0][0]
    assert n == (10 if abs_grad else 9)
    for q, r, row in rows[1:13]:
        value = ROW_VALUES[q][r]
        assert 0 <= row < n, (q, r, row)
        assert value is None or value >= n or row == value, (q, r, row)
    slots = [s[0] for s in rows[13:]]
    for half in (slots[:32], slots[32:]):
        assert sorted(s for s in half if s >= 0) == list(range(9))


def test_a_row_past_the_sums_does_not_build(tmp_path):
    """Nine rows with the deposits of ten."""
    with pytest.raises(RuntimeError, match="every deposit has its row"):
        _run(tmp_path, "raster_slots.h", "", edit=(": 8 - (r >> 1)", ": 8 + (r >> 1)"))


# One block of the binning's passes, reduced to its bookkeeping: rectangle t
# has the words steps[t] (0: a small rectangle or none) and claims[t] tiles. The
# count pass gives the words out in order while they fit; the write pass marks
# the run starts of the rectangles it takes up, and each word up to the last
# marked run's end belongs to the last start at or before it.
REPLAY = """
    const int steps[] = {%s}, claims[] = {%s};
    const int n = sizeof steps / sizeof steps[0];
    int used = 0, ext = 0, owner[kBlockWords] = {}, mark[kBlockWords] = {};
    for (int t = 0; t < n; ++t) {
        uint32_t mask = 0;
        if (steps[t] > 0) {
            if (used + steps[t] <= kBlockWords) {
                mask = kept_mask(used, steps[t], 1 + t %% 64);
                if (kept_rows(mask) != 1 + t %% 64 || kept_steps(mask) != steps[t]) return 1;
                for (int i = 0; i < steps[t]; ++i) owner[used + i] = t + 1;
            }
            used += steps[t] < kBlockWords + 1 ? steps[t] : kBlockWords + 1;
        } else {
            mask = claims[t] > 0;
        }
        if (write_takes(claims[t], mask) && steps[t] > 0 && mask != 0) {
            mark[kept_first(mask)] = t + 1;
            const int end = kept_first(mask) + kept_steps(mask);
            if (end > ext) ext = end;
        }
    }
    for (int i = 0, st = -1; i < ext; ++i) {
        if (mark[i]) st = i;
        std::printf("%%d %%d\\n", owner[i], st < 0 ? -1 : mark[st]);
    }"""

BLOCKS = {
    "first claims nothing": ([3, 5, 1, 0], [0, 40, 7, 9]),
    "one word, nothing": ([1, 1, 1], [0, 0, 2]),
    "one in the middle": ([2, 700, 4], [9, 0, 3]),
    "none claims": ([0, 6, 1], [0, 0, 0]),
    "last does not fit": ([1, 1020, 900, 3], [0, 0, 500, 5]),
    "words to the last": ([1, 1022, 1], [0, 12, 3]),
}


@pytest.mark.parametrize("block", list(BLOCKS))
def test_every_kept_word_lies_in_its_rectangles_run(tmp_path, block):
    steps, claims = BLOCKS[block]
    rows = _run(tmp_path, "bin_words.h",
                REPLAY % (", ".join(map(str, steps)), ", ".join(map(str, claims))))
    assert rows
    assert all(run == own for own, run in rows), "a word in no run, or in another's"


def test_unmarked_runs_without_claims_would_be_found(tmp_path):
    """Taking up only the rectangles that claim tiles leaves words in no run."""
    steps, claims = BLOCKS["first claims nothing"]
    rows = _run(tmp_path, "bin_words.h",
                REPLAY % (", ".join(map(str, steps)), ", ".join(map(str, claims))),
                edit=("return count > 0 || mask != 0u;", "return count > 0;"))
    assert [-1, -1, -1] == [run for own, run in rows if own == 1]
