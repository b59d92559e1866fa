"""Plans and calls on a host-only build of gridgen.cpp and api.cpp (tests/cpp/host_plan.cpp: device memory is host
memory under a byte budget, launches check the tables they would read), for what cannot or must not be
tried on a GPU: tables that a kernel would read through a null pointer, allocations that fail."""
import os
import subprocess

import pytest

import chinium_amd as ca

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.fixture(scope="module")
def host_plan():
    subprocess.run(["make", "-C", CPP, "-s", "host_plan"], check=True)
    return os.path.join(CPP, "host_plan")


@pytest.mark.parametrize("check", ["empty_lists", "failed_plans", "budgets", "planned_again", "reaches"])
def test_host_plan(host_plan, check):
    r = subprocess.run([host_plan, check, ca.DATA_ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
