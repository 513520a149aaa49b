"""Registers of the kernels that are compiled with a model: what the compiler
reports for gfx950, without a device."""
import os
import re
import subprocess

import pytest

from bayadera_amd import build, models

MODELS = {"mvn": models.mvn_model, "diag": models.diag_gaussian_model}


def resources(tmp_path, model, dim, wgs, *defines):
    """{kernel: {"waves": of a SIMD, "scratch": bytes of a lane}}"""
    m = MODELS[model](dim)
    src = tmp_path / "model.hip"
    with open(os.path.join(build.CSRC, "bh_rtc_engine.hip")) as f:
        src.write_text("\n".join(['#include "bh_rtc_prelude.h"', "#pragma clang force_cuda_host_device begin",
                                  *m.source, "#pragma clang force_cuda_host_device end", f.read()]))
    cmd = [build.hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=on",
           "-fhip-fp32-correctly-rounded-divide-sqrt", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "--cuda-device-only", "-c", "-Rpass-analysis=kernel-resource-usage",
           "-I", build.CSRC, f"-DWGS={wgs}", f"-DDIM={dim}", f"-DLOGFN={m.mcmc_logpdf}", *defines,
           str(src), "-o", os.devnull]
    log = subprocess.run(cmd, check=True, capture_output=True, text=True).stderr
    out = {}
    for part in log.split("Function Name: ")[1:]:
        out[part.split()[0]] = {
            "waves": int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", part).group(1)),
            "scratch": int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", part).group(1))}
    return out


# the waves that a half-step without a sample needs to keep: with one fewer,
# 28 coordinates take 12% longer and 38 take 70%
@pytest.mark.parametrize("dim,waves", [(16, 5), (28, 4), (38, 2)])
def test_half_steps_without_a_sample(tmp_path, dim, waves):
    assert resources(tmp_path, "mvn", dim, 256)["bh_stretch_move_bare"]["waves"] >= waves


# a thread of a resident kernel holds a record of each half: 1024 threads leave
# it 128 registers, the 704 that 28 coordinates fit in LDS 168, 384 and fewer 256
@pytest.mark.parametrize("dim,threads", [(16, 1024), (24, 768), (28, 704), (48, 384), (64, 256)])
def test_resident_steps_hold_their_records(tmp_path, dim, threads):
    r = resources(tmp_path, "diag", dim, 64, "-DBH_RESIDENT=1", f"-DBH_RESIDENT_THREADS={threads}")
    assert r["bh_stretch_resident"]["scratch"] == 0 and r["bh_stretch_resident_out"]["scratch"] == 0
