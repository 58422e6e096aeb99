"""The library's kept device blocks (thea_amd/csrc/block_cache.hpp) over a model of the driver: reuse,
bounds, and blocks given back before any allocation fails."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_block_cache(tmp_path):
    exe = tmp_path / "block_cache_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", str(ROOT / "thea_amd" / "csrc"),
                    str(ROOT / "tests" / "block_cache_check.cpp"), "-o", str(exe), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
