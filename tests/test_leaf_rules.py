"""Which kernel the leaves' operators take (p2mOnColumns, l2pSlotsMin in
defmm_amd/csrc/leaf_items.hpp): the plans of few leaves, each of them measured
with both kernels, on which a rule by the mean number of slots alone took the
one that needs 1.3 to 2.5 times as long."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# order, bytes of a real, leaves, slots: whether the matrix cores are faster
L2P = [(2, 8, 125, 2783, 1), (3, 8, 125, 2783, 1), (4, 8, 125, 2783, 1), (5, 8, 149, 1381, 1),
       (6, 8, 125, 2783, 1), (8, 8, 149, 1381, 1), (2, 4, 125, 2783, 1), (3, 4, 149, 1381, 1),
       (5, 4, 149, 1381, 1), (8, 4, 149, 1381, 1), (10, 4, 149, 1381, 1), (9, 4, 160, 160, 1),
       (4, 8, 255, 255, 0), (6, 8, 255, 255, 0), (5, 8, 643, 11445, 0), (6, 4, 985, 8077, 0),
       (8, 8, 821, 7225, 0), (8, 4, 821, 7225, 0), (5, 4, 844, 7850, 1), (6, 8, 988, 16005, 1)]
# order, waves, blocks
P2M = [(2, 160, 160, 1), (2, 651, 651, 1), (3, 847, 958, 1), (4, 4693, 8606, 1), (4, 4693, 4693, 0),
       (5, 1420, 3260, 0), (8, 1420, 3260, 0), (8, 1900, 5000, 1)]


def test_leaf_rules(tmp_path):
    src = tmp_path / "rules.cpp"
    src.write_text('#include <cstdio>\n#include "%s"\nint main() {\n' % os.path.join(
        ROOT, "defmm_amd", "csrc", "leaf_items.hpp") + "".join(
            '  std::printf("%%d\\n", %d >= (long long)dfm::l2pSlotsMin(%d, %d, %d) * %d);\n'
            % (slots, L, size, leaves, leaves) for L, size, leaves, slots, _ in L2P) + "".join(
                '  std::printf("%%d\\n", (int)dfm::p2mOnColumns(%d, false, %d, %d));\n' % t[:3]
                for t in P2M) + "}\n")
    exe = tmp_path / "rules"
    subprocess.check_call(["g++", "-O1", "-std=c++17", str(src), "-o", str(exe)])
    got = [int(x) for x in subprocess.check_output([str(exe)], text=True).split()]
    assert got == [t[-1] for t in L2P + P2M]
