"""Kernel code whose mistakes would reach memory, checked on the host: small programs that
include the kernels' own headers, compiled by hipcc's host pass and run on the CPU."""

import os
import shutil
import subprocess

import pytest

from mingru_amd import build as hip_build

HERE = os.path.dirname(os.path.abspath(__file__))


def _run(name, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    exe = str(tmp_path / name)
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-pthread",
                    "-I", hip_build.CSRC, os.path.join(HERE, name + ".hip"), "-o", exe],
                   check=True, timeout=120)
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60)
    assert res.returncode == 0, res.stdout.decode(errors="replace")


def test_scan_rows_stay_in_the_tensors(tmp_path):
    """Every row the elementwise scans load, steps past the end included, for sequences of
    one step and more."""
    _run("host_rows", tmp_path)


def test_two_buffer_waves_take_the_same_tickets(tmp_path):
    """The persistent form with two row buffers: a wave that reads the shared ticket late
    still takes the workgroup's chunk and not the next one."""
    _run("host_two_buffers", tmp_path)
