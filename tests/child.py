"""Runs a piece of test code in a Python process of its own: for what depends on a
fresh process (memory that a first call takes, calls that a loaded stand-in makes
fail).  One such process at a time."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(code, *args, timeout=100):
    """Runs `code` with `args` as sys.argv[1:]; returns the JSON value on its last line."""
    p = subprocess.run([sys.executable, "-u", "-c", code, *map(str, args)], cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, text=True, timeout=timeout)
    assert p.returncode == 0, f"exit status {p.returncode}\n{p.stdout}\n{p.stderr[-4000:]}"
    return json.loads(p.stdout.strip().splitlines()[-1])
