"""The waits around the last stage of K that are not counts: the transposing kernel's with 2-byte elements, whose last element is
fetched on its own, and the drained prologue of the LDS-transposing form.  The host replay (tests/host_c/mfma_wait_check.cpp)
has to notice each of them missing, one trip late and one trip early."""
import os
import shutil

import pytest

from test_mfma_wait_counts import NEEDED, ROOT, build_and_run

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

EDITS = [
    ("(kbytes & 63) || esz == 2 ? kl - 2", "(kbytes & 63) ? kl - 2"),
    ("(kbytes & 63) || esz == 2 ? kl - 2", "esz == 2 ? kl - 2"),
    ("(kbytes & 63) || esz == 2 ? kl - 2", "(kbytes & 63) || esz == 2 ? kl - 3"),
    ("return mc && kt <= 2;", "return mc && kt <= 1;"),
    ("return mc && kt <= 2;", "return mc && kt <= 3;"),
    ("return mc && kt <= 2;", "return kt <= 2;"),
]


@pytest.mark.parametrize("index", range(len(EDITS)))
def test_an_edited_rule_is_caught(tmp_path, index):
    old, new = EDITS[index]
    for rel in NEEDED:
        dst = tmp_path / rel
        dst.parent.mkdir(parents=True, exist_ok=True)
        shutil.copy(os.path.join(ROOT, rel), dst)
    header = tmp_path / "zluda_amd/csrc/kernels/mfma_wait_counts.hpp"
    text = header.read_text()
    assert text.count(old) == 1, old
    header.write_text(text.replace(old, new))
    res = build_and_run(str(tmp_path), tmp_path, "edit")
    assert res.returncode != 0, "the edit went unnoticed: %s" % new


def test_the_kernels_take_the_rules_from_the_checked_header():
    kernels = os.path.join(ROOT, "zluda_amd", "csrc", "kernels")
    tr = open(os.path.join(kernels, "gemm_mfma_tr.hpp")).read()
    assert tr.count("tail_from = ") == 1 and "tail_from = tr_tail_from(Kl * ESZ, ESZ)" in tr
    assert "if (pipe16_drains_prologue(MC, KT, NSTAGE)) asm volatile(\"s_waitcnt vmcnt(0)\"" in open(os.path.join(kernels, "gemm_mfma_pipe16.hpp")).read()
