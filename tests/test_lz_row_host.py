"""The Lanczos kernels' row product (rcg_lz_row.hpp), which reads eight nonzeros at
a time, on the last rows of an operator with as many nonzeros as 32-bit row
pointers can hold: no index may pass the row's end or wrap.  Compiled for the host
with overflow checks; nothing here runs on a GPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_last_rows_of_the_largest_operator(tmp_path):
    exe = str(tmp_path / "lz_row")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=signed-integer-overflow",
                    "-fno-sanitize-recover=all", os.path.join(HERE, "cpp", "lz_row.cpp"), "-o", exe],
                   check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stderr[-500:]
    x = [1.0, -2.0, 3.0, 0.5]
    rows = [tuple(map(float, line.split())) for line in p.stdout.splitlines()]
    for n, (plain, scaled) in enumerate(rows):
        want = sum(e * x[e % 4] for e in range(1, n + 1))  # exact: small integers and halves
        assert plain == want and scaled == want / 2
    assert len(rows) == 21
