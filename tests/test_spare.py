"""The scratch that the two-launch transforms can do without
(zeknox_amd/csrc/spare.h): on the CPU against an allocator that refuses, and
on the device that a failed allocation gets it back."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle_bind as ob

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "zeknox_amd", "csrc")


def test_refusals_and_drops(tmp_path):
    exe = str(tmp_path / "spare_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "spare_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


@pytest.mark.gpu
def test_a_failed_allocation_gets_the_scratch_back(zk):
    def free_bytes():  # (the HIP runtime that the library is linked to)
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert zk.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    lg, B = 20, 16  # 128 MiB of scratch
    x = ob.canonical(B << lg, 61)
    want = ob.ntt(x, lg, B, False, False)
    buf = zk.DeviceBuffer(B << lg)
    cfg = zk.NTTConfig(batches=B, are_inputs_on_device=True, are_outputs_on_device=True)
    zk._check(zk.lib.zkx_commit_trim(0))
    for _ in range(2):
        buf.copy_from_host(x)
        zk.ntt_batch(0, buf, lg, cfg)
        assert np.array_equal(buf.to_host(), want)
        held = free_bytes()
        with pytest.raises(zk.ZeknoxError):
            zk.DeviceBuffer(1 << 40)  # 8 TiB
        # (the driver's figure moves in steps of its own: half of it shows the free)
        assert free_bytes() >= held + (64 << 20)
