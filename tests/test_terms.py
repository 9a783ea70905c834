"""The sampler's eight-term reads (csrc/wm_terms.h) compiled for the host:
terms below n and zeros from n on, up to the largest n (2^32 - 1)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
BUILD = ROOT / "tests" / "_build"


def test_terms_get8_at_the_ends_of_its_range():
    BUILD.mkdir(exist_ok=True)
    exe = BUILD / "terms_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'project-willamette_amd' / 'csrc'}",
                    str(ROOT / "tests" / "terms_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
