"""The sizes a session takes from its capacity (session_sizes in nh_model.cpp)
against the kernels' rules (nh_forward.hip), over every capacity a session
accepts.  The functions are compiled from the library's sources with g++ (host
code only)."""
import os
import shutil
import subprocess

import pytest

from test_span_runs import SRC, _constant, _grab

CSRC = os.path.dirname(SRC)

MAIN = r"""
int main() {
    const int geoms[][2] = {{12, 2}, {14, 1}, {8, 8}, {6, 3}, {12, 4}};
    for (const auto& g : geoms) {
        Dims D{};
        D.nh = g[0], D.nkv = g[1], D.qk = 48, D.vd = 64;
        const LayerDev L{1024};
        const bool takes = D.nh / D.nkv <= AG_WAVES;
        for (int cap = 1; cap <= 1 << 20; cap += cap < 64900 ? 401 : cap < 65600 ? 1 : 65521) {
            session_sizes(D, cap);
            // capacities whose positions alone fit 16 bits of value stride
            if (takes && (cap + 4 + 15) / 16 * 16 < 65536 && !attend_group_fits(D, L)) {
                std::printf("capacity %d of %d heads: no grouped attention (stride %d)\n", cap, g[0], D.vcap);
                return 1;
            }
            // the packed argument gives the stride back
            const int wv = (int)((unsigned)L.window | (unsigned)(D.vcap / 16) << 16);
            if (attend_group_fits(D, L) && (int)((unsigned)wv >> 16) * 16 != D.vcap) return 2;
            if (D.vcap < D.kslots + 4 || D.kslots < D.stage0 + D.batch || D.stage0 < cap || D.batch % 64) return 3;
        }
    }
    std::printf("ok\n");
    return 0;
}
"""


def compile_and_run(tmp_path, main):
    src = open(SRC).read()
    hdr = open(os.path.join(CSRC, "nh_forward.h")).read()
    mod = open(os.path.join(CSRC, "nh_model.cpp")).read()
    code = "".join([
        "#include <algorithm>\n#include <cstddef>\n#include <cstdint>\n#include <cstdio>\n",
        "using std::min; using std::max;\nnamespace nh {\n",
        "constexpr int BATCH_MIN = 512, BATCH_MAX = 2048;\n",
        _constant(hdr, "ATT_CHUNK_MAX"),
        _constant(src, "NATIVE_TEAM"), _constant(src, "AG_WAVES"), _grab(hdr, "struct Dims {", "\n};\n"),
        "struct LayerDev { int window; };\n",
        _grab(src, "static bool attend_group_fits("),
        _grab(src, "__host__ __device__ inline void key_chunks("),
        "}\nusing namespace nh;\n",
        _grab(mod, "size_t round_up(", "}\n"),
        _grab(mod, "int key_chunk_count("),
        _grab(mod, "int feed_chunks(", "}\n"),
        _grab(mod, "void session_sizes("),
        main,
    ]).replace("__host__ __device__ inline", "inline")
    assert "constexpr int BATCH_MIN = 512, BATCH_MAX = 2048;" in hdr
    cpp, exe = tmp_path / "sizes.cpp", tmp_path / "sizes"
    cpp.write_text(code)
    subprocess.run(["g++", "-O1", "-std=c++17", str(cpp), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "ok" in r.stdout


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_capacity_keeps_grouped_attention(tmp_path):
    """The staging slots behind a capacity's own take no capacity off the
    grouped attention kernel."""
    compile_and_run(tmp_path, MAIN)


CHUNKS = r"""
int main() {
    // a feed's rows (nested chunks): every count of keys up to the capacity
    // fits the partials a row has room for, and some count fills them
    for (int nkv = 1; nkv <= 8; ++nkv) {
        int most = 0, count, size;
        for (int n = 1; n <= 40000; ++n) {
            key_chunks(n, nkv, true, count, size);
            if (size > 256) return 1;
            most = std::max(most, count);
            if (most > feed_chunks(n)) { std::printf("%d keys: %d chunks\n", n, most); return 2; }
            if (n % 256 == 0 && most != feed_chunks(n)) { std::printf("%d keys: %d of %d\n", n, most, feed_chunks(n)); return 3; }
        }
    }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_feed_chunks(tmp_path):
    """The chunk partials of a feed's rows hold what their keys need, not a
    step's finer split."""
    compile_and_run(tmp_path, CHUNKS)
