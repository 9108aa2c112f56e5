"""The result slots of the separate routines (csrc/omhd_slot.h) after calls
that end on an error: a slot is given back clean or not at all.  Runs on a
stand-in for the HIP calls (tests/native/slotcheck.cpp)."""
import subprocess
import sys
from pathlib import Path

import pytest

from omhd_testlib import NATIVE_DIR, SANITIZED

SO = NATIVE_DIR / "libslotcheck.so"
SLOTS = 64


def run(code):
    """In a process of its own: the slots are the process's."""
    if not SO.exists():
        d = Path(__file__).resolve().parent / "native"
        subprocess.run(["make", "-s", "-C", str(d)] + (["sanitize"] if SANITIZED else []), check=True)
    subprocess.run([sys.executable, "-c", f"import ctypes; L = ctypes.CDLL({str(SO)!r})\n" + code], check=True,
                   timeout=60)


@pytest.mark.parametrize("calls", (1, 3, SLOTS + 5))
def test_a_broken_call_leaves_its_slot_clean(calls):
    run(f"L.slotc_break({calls}, 0)\nassert L.slotc_take_all({SLOTS}) == {SLOTS}")


def test_a_slot_that_cannot_be_cleared_is_given_up():
    run(f"L.slotc_break(3, 3)\nassert L.slotc_take_all({SLOTS} - 3) == {SLOTS} - 3\nassert L.slotc_acquire() == 0")


def test_a_call_does_not_wait_for_slots_that_were_given_up():
    run(f"L.slotc_break({SLOTS}, {SLOTS})\nassert L.slotc_take_all(1) == 0\nassert L.slotc_acquire() != 0")


def test_more_threads_than_slots():
    run("assert L.slotc_threads(80, 40) == 0")
