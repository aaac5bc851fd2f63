"""A line within one tile takes the count pass's short way (rzg::single_tile);
this CPU test (tests/cpu_single_tile.cpp) requires of it exactly the record,
bit for bit, that the step-by-step decomposition makes, on lines of 0.03 to 10
px that start on, beside and between tile and pixel edges, in every grid phase
and edge mode."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_single_tile_is_the_decomposition(tmp_path):
    exe = str(tmp_path / "cpu_single_tile")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "cpu_single_tile.cpp")], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
