"""rzg::ae_piece walks only the rows of an edge that can come out left of x = 0;
this CPU test (tests/cpu_ae_walk.cpp) compares its vertices bit for bit with
those of the walk over every row."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_short_walk_is_the_whole_walk(tmp_path):
    exe = str(tmp_path / "cpu_ae_walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "cpu_ae_walk.cpp")], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
