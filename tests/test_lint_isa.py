"""The assembly check of the build: counted waits of the tile kernels' ring loop, on listings written out here."""
import importlib.util
from pathlib import Path

import pytest

_SPEC = importlib.util.spec_from_file_location(
    "lint_isa", Path(__file__).resolve().parents[1] / "tyloquant_amd" / "csrc" / "lint_isa.py")
lint_isa = importlib.util.module_from_spec(_SPEC)
_SPEC.loader.exec_module(lint_isa)

NAME = "_ZN3mfq15row_tile_kernelILi0ELi8ELi8ELi2ELi4EEEvNS_11RowTileArgsEii"   # R = 4
COPY, LOAD, MFMA = "buffer_load_dwordx4 v1, s[16:19], s5 offen lds", "buffer_load_dwordx4 v[2:5], v6, s[12:15], s5 offen", "v_mfma_f32_16x16x32_f16 a, b"


def _listing(intervals, wait, prologue_wait="s_waitcnt vmcnt(0) lgkmcnt(0)", name=NAME):
    """A kernel of that many stages per pass: each a wait, a barrier and the requests of the interval."""
    body = [COPY] * 6 + [prologue_wait, "s_barrier", ".LBB0_3:"]
    for requests in intervals:
        body += [f"s_waitcnt vmcnt({wait})", "s_barrier", *requests, MFMA]
    body += ["s_cbranch_scc1 .LBB0_3", "s_waitcnt vmcnt(0)", "s_barrier", "s_endpgm"]
    return "\n".join([f"{name}: ; @x", *("\t" + b if not b.endswith(":") else b for b in body), ".Lfunc_end0:"]) + "\n"


def _lint(tmp_path, text):
    f = tmp_path / "k.s"
    f.write_text(text)
    return lint_isa.lint_tiles(str(f))


IN_ORDER = [COPY, COPY, LOAD, LOAD, LOAD, LOAD]
SWAPPED = [COPY, LOAD, LOAD, COPY, LOAD, LOAD]      # two weight requests ahead of the last copy


def test_requests_in_source_order_pass(tmp_path):
    errors, seen = _lint(tmp_path, _listing([IN_ORDER] * 4, 10))     # two intervals later ten requests are younger
    assert seen == 1 and not errors


def test_a_copy_behind_a_weight_request_fails(tmp_path):
    """Eight requests younger than the copy, ten admitted: the barrier two intervals later does not cover it."""
    errors, _ = _lint(tmp_path, _listing([IN_ORDER, SWAPPED, IN_ORDER, IN_ORDER], 10))
    assert len(errors) == 1 and "barrier 4 of 4" in errors[0] and "1 of 2" in errors[0]
    assert not _lint(tmp_path, _listing([IN_ORDER, SWAPPED, IN_ORDER, IN_ORDER], 8))[0]


@pytest.mark.parametrize("wait,ok", [(9, True), (10, True), (11, False)])
def test_the_wait_may_admit_as_many_requests_as_are_younger(tmp_path, wait, ok):
    assert bool(_lint(tmp_path, _listing([IN_ORDER] * 2, wait))[0]) != ok


def test_a_copy_on_the_wrong_side_of_a_barrier_fails(tmp_path):
    errors, _ = _lint(tmp_path, _listing([IN_ORDER + [COPY], IN_ORDER[1:]], 2))
    assert errors and "copies per barrier interval" in errors[0]


def test_spilled_registers_in_a_ring_loop_fail(tmp_path):
    reload = "scratch_load_dword v7, off, off offset:8"
    errors, _ = _lint(tmp_path, _listing([IN_ORDER, IN_ORDER + [reload]], 8))
    assert errors == [f"{tmp_path / 'k.s'}: {NAME}: 1 scratch accesses in a ring loop"]
    outside = _listing([IN_ORDER] * 2, 10).replace("\ts_endpgm", f"\t{reload}\n\ts_endpgm")
    assert reload in outside and not _lint(tmp_path, outside)[0]


def test_first_stages_need_a_full_wait(tmp_path):
    errors, _ = _lint(tmp_path, _listing([IN_ORDER] * 4, 10, prologue_wait="s_waitcnt vmcnt(2)"))
    assert errors and "without vmcnt(0)" in errors[0]


def test_every_ring_loop_of_a_kernel_with_several_is_read(tmp_path):
    """The kernel of routed experts holds a loop per chunk size, and loops over group sums that wait for their copies on the spot."""
    name = "_ZN3mfq15moe_tile_kernelILb1EEEvNS_11MoeTileArgsE"
    def kernel(second):
        one = _listing([IN_ORDER] * 4, 10, name=name).split("\n")
        two = _listing(second, 10, name=name).replace(".LBB0_3", ".LBB0_5").split("\n")
        sums = ["\t.LBB0_2:".strip(), f"\t{COPY}", "\ts_waitcnt vmcnt(0)", "\ts_barrier", f"\t{MFMA}", "\ts_cbranch_scc1 .LBB0_2"]
        return "\n".join(one[:1] + sums + one[1:-2] + two[1:])
    assert _lint(tmp_path, kernel([IN_ORDER] * 4)) == ([], 1)
    errors, _ = _lint(tmp_path, kernel([IN_ORDER, SWAPPED, IN_ORDER, IN_ORDER]))
    assert len(errors) == 1 and "barrier 4 of 4" in errors[0]


def test_a_tile_kernel_it_cannot_read_is_an_error(tmp_path):
    errors, seen = _lint(tmp_path, _listing([IN_ORDER] * 4, 10, name="_ZN3mfq15row_tile_kernelILi0ELi8EEEvv"))
    assert errors and seen == 0


def test_a_block_moved_out_of_line_is_not_taken_for_the_ring_loop(tmp_path):
    """A block behind the kernel's end that jumps back to in front of the loop spans more than the loop."""
    text = _listing([IN_ORDER] * 4, 10).replace("\ts_endpgm", f"\ts_endpgm\n.LBB0_9:\n\t{MFMA}\n\ts_branch .LBB0_1").replace(
        ".LBB0_3:", ".LBB0_1:\n.LBB0_3:", 1)
    errors, seen = _lint(tmp_path, text)
    assert seen == 1 and not errors
