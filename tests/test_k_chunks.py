"""How K is cut into chunks and slices (cuda_hgemm_amd/csrc/k_chunks.h), checked on the CPU up to the largest K a call may
have (2^31 - 1 elements per operand, so M = N = 1)."""
import os
import subprocess
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "cuda_hgemm_amd", "csrc", "k_chunks.h")

PROGRAM = textwrap.dedent(
    r"""
    #include "%s"
    #include <cstdio>
    using namespace hgemm;
    static bool check(long long K) {
        for (int bk = 32; bk <= 64; bk *= 2) {
            const int chunks = chunks_of((int)K, bk);
            if ((long long)chunks * bk < K || (long long)(chunks - 1) * bk >= K) return printf("chunks: K %%lld\n", K), false;
            if (K %% 8 == 0 && tail_pieces((int)K, bk) * 8 != (long long)chunks * bk - K) return printf("tail: K %%lld\n", K), false;
            for (int slices = 1; slices <= 32 && slices <= chunks; ++slices) {
                int next = 0;
                for (int s = 0; s < slices; ++s) {
                    int first, count;
                    slice_of_k(chunks, slices, s, first, count);
                    if (first != next || count < chunks / slices || count > chunks / slices + 1) return printf("slice: K %%lld\n", K), false;
                    next = first + count;
                }
                if (next != chunks) return printf("slices: K %%lld\n", K), false;
            }
        }
        return true;
    }
    int main() {
        for (long long K = 1; K <= 5000; ++K)
            if (!check(K)) return 1;
        for (long long K = (1ll << 31) - 300; K < (1ll << 31); ++K)
            if (!check(K)) return 1;
        return printf("ok\n"), 0;
    }
    """
)


def test_chunks_and_slices_cover_k(tmp_path):
    src, exe = tmp_path / "k_chunks.cpp", tmp_path / "k_chunks"
    src.write_text(PROGRAM % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(exe), str(src)],
                   check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
