"""The library where memory runs out: device allocations refused from a given
total on, pinned host memory refused altogether (tests/mem_child.py)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "mem_child.py")


def _run(scenario):
    r = subprocess.run([sys.executable, "-u", CHILD, scenario], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


@pytest.mark.parametrize("scenario", ["create_at_the_limit", "contacts_at_the_limit"])
def test_a_refused_allocation_leaves_nothing_behind(scenario):
    _run(scenario)


def test_results_without_pinned_memory():
    _run("no_pinned_memory")


def test_memory_of_one_instance_serves_the_next():
    _run("another_instance")


def test_lists_give_way():
    _run("lists_make_room")


def test_small_handles_take_few_allocations():
    _run("small_handles")
