"""What the row-split FP64 kernel (prune_fp64r.hip) reads for a step of a tree's
program lies inside the tree's transition matrices, down to two leaves."""
import os
import subprocess


def test_steps_read_branches_of_the_tree(tmp_path):
    src = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "phylocsf_amd", "csrc")
    exe = str(tmp_path / "step_branch")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + src, "-I" + os.path.join(src, "host"), "-o", exe,
                    os.path.join(os.path.dirname(os.path.abspath(__file__)), "step_branch.cpp"),
                    os.path.join(src, "host", "program.cpp")], check=True)
    rows = [tuple(map(int, ln.split())) for ln in
            subprocess.run([exe], check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()]
    assert len(rows) == 78
    assert all(top < branches for _, branches, top in rows)
