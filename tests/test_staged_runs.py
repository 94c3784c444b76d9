"""The staged form of a feed under an attention span (staged_range and
staged_runs in nh_forward.hip) against the general path's key mapping, chunk by
chunk (slot_of(span_key(...)) over the live runs, infer.rs:1749-1826), on
random sinks, rings, windows, feeds and key chunk sizes: every key of every
row must be the same position, found through its run in a slot that holds it,
with value columns that do not overlap; and the slots the feed leaves behind
must be those of feeding it chunk by chunk.  The functions are compiled from the
library's source with g++ (host code only)."""
import os
import shutil
import subprocess

import pytest

from test_span_runs import SRC, _constant, _grab

HARNESS = r"""
int main() {
    std::mt19937 rng(11);
    long rows_seen = 0, keys = 0, multi = 0;
    for (int it = 0; it < 1500; ++it) {
        Dims D{};
        D.sink = rng() % 3 ? (int)(rng() % 150) : 0;
        D.ring = FWD_ROWS + (int)(rng() % 300);
        const int p0 = rng() % 3 ? (int)(rng() % 500) : 0, rows = 2 + (int)(rng() % 300);
        if (rows % FWD_ROWS == 1) continue;  // a one-token chunk is a step
        const int cap = p0 + rows;
        D.stage0 = (cap + 15) / 16 * 16;
        const int window = rng() % 2 ? 0 : 1 + (int)(rng() % 400);
        const int chunk = 16 * (1 + (int)(rng() % 16));
        std::vector<int> slots(D.stage0 + 512, -1), ref;
        for (int p = 0; p < p0; ++p) slots[slot_of(D, p)] = p;
        ref = slots;
        for (int r = 0; r < rows; ++r) slots[D.stage0 + r] = p0 + r;
        for (int c0 = 0; c0 < rows; c0 += FWD_ROWS) {
            const int end = p0 + std::min(rows, c0 + FWD_ROWS);
            for (int p = p0 + c0; p < end; ++p) ref[slot_of(D, p)] = p;
            // the live runs of the chunk (span_keys)
            KeySpan K{};
            K.end = end;
            auto scan = [&](int lo, int hi) {
                for (int p = lo, a = -1; p <= hi; ++p) {
                    const bool ok = p < hi && ref[slot_of(D, p)] == p;
                    if (ok && a < 0) a = p;
                    if (!ok && a >= 0) K.lo[K.nrun] = a, K.hi[K.nrun] = p, ++K.nrun, a = -1;
                }
            };
            scan(0, std::min(D.sink, end));
            scan(std::max(std::max(end - D.ring, D.sink), std::min(D.sink, end)), end);
            for (int row = c0; row < end - p0; ++row) {
                const int pos = p0 + row, lo = window > 0 && pos + 1 > window ? pos + 1 - window : 0;
                int alo, ahi, blo, bhi, ahi2, blo2, n = 0;
                span_ranges(D, K, lo, pos, alo, ahi, blo, bhi);
                for (int r = 0; r < K.nrun; ++r)
                    n += span_overlap(K.lo[r], K.hi[r], alo, ahi) + span_overlap(K.lo[r], K.hi[r], blo, bhi);
                const int n2 = staged_range(D, p0, rows, row, lo, ahi2, blo2);
                if (n2 != n) { std::printf("case %d row %d: %d keys, want %d\n", it, row, n2, n); return 1; }
                ++rows_seen;
                for (int k0 = 0; k0 < n; k0 += chunk) {
                    const int len = std::min(chunk, n - k0);
                    StagedRuns R;
                    staged_runs(D, p0, pos, lo, ahi2, blo2, k0, k0 + len, R);
                    std::vector<char> used(384, 0);
                    if (R.cols > 384 || R.cols % 16) { std::printf("case %d: %d columns\n", it, R.cols); return 1; }
                    multi += R.key[2] < len;
                    for (int i = 0; i < len; ++i) {
                        int r = 0;
                        while (r + 1 < AG_RUNS && i >= R.key[r + 1]) ++r;
                        const int slot = R.slot[r] + i - R.key[r], col = R.col[r] + (R.slot[r] & 15) + i - R.key[r];
                        const int want = span_key(K, alo, ahi, blo, bhi, k0 + i);
                        // (the 16-byte chunk the column is staged from)
                        const int rr = col >= R.col[3] ? 3 : col >= R.col[2] ? 2 : col >= R.col[1] ? 1 : 0;
                        const int from = (R.slot[rr] & ~15) + col - R.col[rr];
                        if (slot < 0 || slot >= (int)slots.size() || slots[slot] != want || from != slot || col < 0 ||
                            col >= R.cols || used[col]) {
                            std::printf("case %d row %d key %d: slot %d, position %d\n", it, row, k0 + i, slot, want);
                            return 1;
                        }
                        used[col] = 1;
                        ++keys;
                    }
                }
            }
        }
        for (int r = 0; r < rows; ++r) {
            const int p = p0 + r;
            if (p < D.sink || p + D.ring >= p0 + rows) slots[slot_of(D, p)] = p;
        }
        for (int i = 0; i < D.stage0; ++i)
            if (slots[i] != ref[i]) { std::printf("case %d: slot %d holds %d, want %d\n", it, i, slots[i], ref[i]); return 1; }
    }
    std::printf("rows %ld keys %ld, %ld chunks of three runs or more, ok\n", rows_seen, keys, multi);
    return rows_seen > 100000 && multi > 1000 ? 0 : 2;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_staged_runs_match_chunk_by_chunk(tmp_path):
    src = open(SRC).read()
    hdr = open(os.path.join(os.path.dirname(SRC), "nh_forward.h")).read()
    code = "".join([
        "#include <algorithm>\n#include <cstdio>\n#include <random>\n#include <vector>\nusing std::min; using std::max;\n",
        _constant(hdr, "SPAN_RUNS"), _constant(hdr, "FWD_ROWS"), _constant(hdr, "ATT_CHUNK_MAX"),
        _constant(src, "AG_RUNS"),
        "struct Dims { int sink, ring, stage0; };\n",
        "struct KeySpan { int end; int nrun; int lo[SPAN_RUNS], hi[SPAN_RUNS]; };\n",
        _grab(src, "struct StagedRuns {", "\n};\n"),
        _grab(src, "__host__ __device__ inline void span_ranges("),
        _grab(src, "__host__ __device__ inline int span_overlap("),
        _grab(src, "__device__ __forceinline__ int span_key("),
        _grab(src, "__device__ __forceinline__ int slot_of("),
        _grab(src, "__host__ __device__ inline int staged_range("),
        _grab(src, "__host__ __device__ inline void staged_runs("),
        HARNESS,
    ]).replace("__host__ __device__ inline", "inline").replace("__device__ __forceinline__", "inline")
    cpp = tmp_path / "staged.cpp"
    cpp.write_text(code)
    exe = tmp_path / "staged"
    subprocess.run(["g++", "-O1", "-std=c++17", str(cpp), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "ok" in r.stdout
