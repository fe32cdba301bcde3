"""The autotuner's choice of the predictor schedule from its trials' times: the
split only where it is clearly faster than the one kernel."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pypde_amd", "csrc")


def test_ties_go_to_the_one_kernel(tmp_path):
    main = tmp_path / "choice.cpp"
    main.write_text('#include <cstdio>\n#include <cstdlib>\n#include "tune.h"\n'
                    "int main(int n, char** a) {\n"
                    "  double t[8];\n  for (int i = 1; i < n; i++) t[i - 1] = atof(a[i]);\n"
                    '  printf("%d %d\\n", pypde::fastest(t, n - 1),\n'
                    "         pypde::predictor_schedule(t, n - 1));\n}\n")
    exe = str(tmp_path / "choice")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", exe, str(main)], check=True)

    def choose(*ms):
        out = subprocess.run([exe] + [str(x) for x in ms], check=True, capture_output=True,
                             text=True).stdout
        return tuple(int(x) for x in out.split())

    assert choose(0.1566, 0.1563, 0.17) == (1, 0)     # a tie
    assert choose(1.0, 0.96, 0.951) == (2, 0)         # faster, not clearly
    assert choose(1.0, 0.96, 0.94) == (2, 2)
    assert choose(1.0, 0.8, 0.94) == (1, 1)
    assert choose(0.4, 0.47, 0.45) == (0, 0)
    assert choose(0.3) == (0, 0)                      # one schedule only
    assert choose(1e30, 1e30, 1e30) == (0, 0)         # no trial was timed
