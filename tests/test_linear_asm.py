"""The LayerNorm-Linear band form's loads to LDS, in the generated gfx950 code (CPU only, needs only hipcc).

The kernel waits by counting its loads in flight, which is right only for one order of them. In the loop
scheduling barriers keep that order; before it, an explicit wait has to leave nothing in flight but x of the
two steps that are multiplied last, so that the weight of the first step is in LDS whatever order the
compiler chose."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "cti-inference-optimization_amd", "csrc", "ebag_linear.hip")
X_LOADS = 2  # x loads per thread and step (128 rows of 64 by 512 threads, 16 bytes each)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "linear.s"
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-ffp-contract=off", f"-I{ROOT}/include", "--cuda-device-only", "-S",
                    SOURCE, "-o", str(out)], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    found = re.findall(r"^(_ZN\S*ln_linear_band_kernel\S*):(.*?)s_endpgm", out.read_text(), re.S | re.M)
    assert len(found) == 9  # three widths; plain, fp32 and bf16 parameters
    return found


def _events(body):
    """The loads, vmcnt waits and barriers up to the first product, in program order."""
    for line in body.splitlines():
        line = line.strip()
        if line.startswith("v_mfma"):
            return
        if line.startswith(("buffer_load", "global_load")):
            yield "weight" if line.endswith(" lds") else "load", 0
        elif line.startswith("s_waitcnt") and "vmcnt" in line:
            yield "wait", int(re.search(r"vmcnt\((\d+)\)", line).group(1))
        elif line.startswith("s_barrier"):
            yield "barrier", 0


def test_the_first_weights_are_waited_for_before_the_loop(kernels):
    for name, body in kernels:
        events = list(_events(body))
        last = max(i for i, (what, _) in enumerate(events) if what == "barrier")
        assert sum(what == "weight" for what, _ in events[:last]) in (4, 6, 8), name  # both halves of step 0
        flight, waited = [], None
        for what, n in events[:last]:
            if what == "wait":
                flight = flight[len(flight) - min(n, len(flight)):]
                waited = n
            elif what != "barrier":
                flight.append(what)
                waited = None
        assert flight == ["load"] * (2 * X_LOADS), name
        assert waited == 2 * X_LOADS, f"{name}: no wait for the weight between the last load and the loop"
