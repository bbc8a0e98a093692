"""Sources that instantiate the tracked walk are compiled with NaN semantics: the
walk retires lanes by NaN plane parameters."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "framelab_amd", "csrc")
BLIND = ("-fno-honor-nans", "-ffast-math", "-ffinite-math-only", "-menable-no-nans")


def test_walks_keep_nan_semantics():
    lines = subprocess.run(["make", "-n", "-B", "-C", CSRC], check=True, capture_output=True, text=True).stdout.splitlines()
    commands = {m.group(1): line for line in lines if (m := re.search(r"(\w+)\.hip$", line.strip()))}
    walks = [n for n in commands if re.search(r"\b(walk_rays|fl_fan_ray_sum)\b", open(os.path.join(CSRC, n + ".hip")).read())]
    assert {"siddon", "batch"} <= set(walks)
    for name in walks:
        assert not any(flag in commands[name].split() for flag in BLIND), name
