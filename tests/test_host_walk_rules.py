"""The walk's size rules, without a GPU: which trees may be walked at 32-bit byte
offsets, by how many lanes, and where a chunk's walk is shared.
tests/cpp/walk_rules_main.cpp holds the checks; __graft_entry__.build() compiles it."""
import os
import subprocess

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "hbt_rules_test")


def test_walk_rules_on_the_host():
    assert os.path.exists(EXE), f"{EXE} is missing: build it with __graft_entry__.build()"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
