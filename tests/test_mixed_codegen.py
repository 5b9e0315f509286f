"""The generated gfx950 code of the mixed-radix, chirp-z and ragged kernels, on the CPU: each source is
compiled to device assembly with the library's own flags, and no kernel may keep more in scratch memory than
is known and measured to be worth it."""
import concurrent.futures
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "accelerate-fft_amd"))

SOURCES = ["afft_mixed_f32", "afft_mixed_f64", "afft_chirpz_f32", "afft_chirpz_f64", "afft_wide_f32", "afft_wide_f64",
           "afft_ragged"]

# bytes a lane: <Real, EMAX, ROWS, BLUE>
ALLOWED = {
    "afft_mixedIfLi31ELb0ELb0EE": 48,  # butterflies of 31 in 128 registers
    "afft_mixedIdLi16ELb0ELb1EE": 24,
}


@pytest.fixture(scope="module")
def private_bytes(tmp_path_factory):
    import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("asm")

    def compile_one(name):
        asm = str(out / (name + ".s"))
        flags = [f for f in build.COMMON if f != "-fPIC"]
        r = subprocess.run([build.HIPCC] + flags + ["-S", "--cuda-device-only", os.path.join(build.CSRC, name + ".hip"),
                                                    "-o", asm], capture_output=True, text=True, timeout=900)
        assert r.returncode == 0, r.stderr[-2000:]
        with open(asm) as f:
            text = f.read()
        return re.findall(r"\.name:\s+(_ZN4afft\w+)\n\s+\.private_segment_fixed_size:\s+(\d+)", text)

    with concurrent.futures.ThreadPoolExecutor(max_workers=7) as ex:
        return {k: int(v) for found in ex.map(compile_one, SOURCES) for k, v in found}


def test_scratch_memory_of_the_mixed_kernels(private_bytes):
    assert len(private_bytes) == 2 * (4 + 4 + 2 + 2)
    for name, size in private_bytes.items():
        limit = max((v for k, v in ALLOWED.items() if k in name), default=0)
        assert size <= limit, f"{name}: {size} bytes of scratch memory a lane"
