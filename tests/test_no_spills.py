"""Registers of the long prompt's projection kernels (csrc/qkv_prefill.hip), from the
compiler's own report: accumulators take most of them, and an epilogue that spills
costs the fused 256 x 384 tiles 3-4 % of their time."""
import pathlib
import re
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "llm-inference_amd" / "csrc"


def test_projection_kernels_do_not_spill(tmp_path):
    # the build's own command line for this file
    out = subprocess.run(["make", "-C", str(CSRC), "-n", "-B", "../lib/obj/qkv_prefill.o"],
                         capture_output=True, text=True, check=True).stdout
    line = next(x for x in out.splitlines() if "-c qkv_prefill.hip" in x)
    line = re.sub(r"-o \S+", f"-o {tmp_path / 'x.o'}", line)
    r = subprocess.run(line + " -Rpass-analysis=kernel-resource-usage", shell=True, cwd=CSRC,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    names = re.findall(r"Function Name: (\S+)", r.stderr)
    spills = [int(x) for x in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    assert len(names) == len(spills) >= 10, r.stderr[-2000:]
    assert not any(spills), dict(zip(names, spills))
