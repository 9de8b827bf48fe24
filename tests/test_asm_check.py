"""The build check of the tiled GEMM's inline LDS reads (CPU only): the checker
flags a planted use of an in-flight read register, passes the clean form, and
passes the library's own device assembly."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "ane-training_amd")
sys.path.insert(0, PKG)

import check_lds_asm  # noqa: E402
import pytest  # noqa: E402

HEAD = "_Z11k_gemm_tileILi64ELi64ELi0EEvPKtiS1_i7EpiArgsii:\n"
TAIL = ".Lfunc_end0:\n"


def test_flags_planted_use_of_pending_register():
    asm = HEAD + ("\tds_read_b128 v[4:7], v1\n"
                  "\tv_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]\n"
                  "\ts_waitcnt lgkmcnt(0)\n") + TAIL
    names, bad = check_lds_asm.check(asm)
    assert len(names) == 1 and len(bad) == 1


def test_flags_copy_of_pending_register():
    asm = HEAD + ("\tds_read_b128 v[4:7], v1\n"
                  "\tv_mov_b32 v20, v5\n"
                  "\ts_waitcnt lgkmcnt(0)\n") + TAIL
    assert len(check_lds_asm.check(asm)[1]) == 1


@pytest.mark.parametrize("op", ["ds_write_b32 v1, v5", "ds_write_b32 v4, v2", "ds_read_b32 v20, v6"])
def test_flags_lds_operation_on_pending_register(op):
    """As data, and as the address of a write or another read."""
    asm = HEAD + f"\tds_read_b128 v[4:7], v1\n\t{op}\n\ts_waitcnt lgkmcnt(0)\n" + TAIL
    assert len(check_lds_asm.check(asm)[1]) == 1


def test_passes_use_after_wait_and_unrelated_work():
    asm = HEAD + ("\tds_read_b128 v[4:7], v1\n"
                  "\tv_mfma_f32_32x32x16_f16 a[16:31], v[12:15], v[8:11], a[16:31]\n"
                  "\ts_waitcnt lgkmcnt(0)\n"
                  "\tv_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]\n") + TAIL
    names, bad = check_lds_asm.check(asm)
    assert len(names) == 1 and not bad


def test_partial_wait_retires_only_older_reads():
    """lgkmcnt(1) after two LDS reads retires the older one only (LDS operations
    complete in order)."""
    two = "\tds_read_b128 v[4:7], v1\n\tds_read_b128 v[8:11], v1 offset:32\n\ts_waitcnt lgkmcnt(1)\n"
    assert not check_lds_asm.check(HEAD + two + "\tv_mul_f32_e32 v20, v4, v20\n" + TAIL)[1]
    assert len(check_lds_asm.check(HEAD + two + "\tv_mul_f32_e32 v20, v8, v20\n" + TAIL)[1]) == 1


def test_partial_wait_with_scalar_load_retires_nothing():
    """A scalar load in flight can complete out of order: lgkmcnt(1) then
    retires no LDS read."""
    asm = HEAD + ("\tds_read_b128 v[4:7], v1\n"
                  "\ts_load_dwordx2 s[0:1], s[4:5], 0x0\n"
                  "\ts_waitcnt lgkmcnt(1)\n"
                  "\tv_mul_f32_e32 v20, v4, v20\n") + TAIL
    assert len(check_lds_asm.check(asm)[1]) == 1


WRITE = "\tds_write_b32 v1, v2\n"


@pytest.mark.parametrize("n", [3, 63, 64, 65, 200])
def test_read_stays_pending_behind_any_number_of_writes(n):
    """Operations that nothing has waited for retire no read before them; a
    partial wait that leaves fewer than them in flight does."""
    read, use = "\tds_read_b128 v[4:7], v1\n", "\tv_mul_f32_e32 v20, v4, v20\n"
    assert len(check_lds_asm.check(HEAD + read + n * WRITE + use + TAIL)[1]) == 1
    assert not check_lds_asm.check(HEAD + read + n * WRITE + "\ts_waitcnt lgkmcnt(3)\n" + use + TAIL)[1]


@pytest.mark.parametrize("n", [1, 64, 200])
def test_scalar_load_stays_in_flight_behind_any_number_of_writes(n):
    asm = HEAD + ("\ts_load_dwordx2 s[0:1], s[4:5], 0x0\n" + n * WRITE + "\tds_read_b128 v[4:7], v1\n" + WRITE +
                  "\ts_waitcnt lgkmcnt(1)\n"
                  "\tv_mul_f32_e32 v20, v4, v20\n") + TAIL
    assert len(check_lds_asm.check(asm)[1]) == 1


def _loop(body, exit_block="", after=""):
    """A loop whose text holds exit_block (entered from its head, back to its
    end) before the back edge, as the compiler places rare blocks."""
    return HEAD + ("\ts_mov_b32 s0, 0\n"
                   ".LBB0_1:\n" + body +
                   "\ts_cbranch_vccnz .LBB0_3\n"
                   "\ts_branch .LBB0_2\n"
                   ".LBB0_3:\n" + exit_block +
                   "\ts_branch .LBB0_4\n"
                   ".LBB0_2:\n"
                   "\ts_cbranch_scc1 .LBB0_1\n"
                   ".LBB0_4:\n" + after + "\ts_endpgm\n") + TAIL


READ, USE, WAIT = "\tds_read_b128 v[4:7], v1\n", "\tv_mul_f32_e32 v20, v4, v20\n", "\ts_waitcnt lgkmcnt(0)\n"


def test_pending_read_is_followed_along_branches():
    # over a forward branch into the block that uses it
    assert len(check_lds_asm.check(_loop(READ, after=USE))[1]) == 1
    assert not check_lds_asm.check(_loop(READ + WAIT, after=USE))[1]
    # round the back edge: read at the end of one trip, used at the head of the next
    assert len(check_lds_asm.check(_loop(USE + READ))[1]) == 1
    assert not check_lds_asm.check(_loop(WAIT + USE + READ))[1]
    # a wait in the block that only the exit takes retires nothing in the loop
    assert len(check_lds_asm.check(_loop(USE + READ, exit_block=WAIT))[1]) == 1
    # the exit's own read is not in flight in the loop that its text interrupts
    assert not check_lds_asm.check(_loop("\tv_mul_f32_e32 v20, v4, v20\n", exit_block=READ + WAIT))[1]
    # used on one side of a branch alone
    assert len(check_lds_asm.check(_loop(READ, exit_block=USE, after=WAIT))[1]) == 1


def test_loop_of_writes_without_a_wait_ends():
    assert not check_lds_asm.check(_loop(3 * WRITE, after=WAIT))[1]
    assert len(check_lds_asm.check(_loop(3 * WRITE + READ, after=USE))[1]) == 1


@pytest.mark.skipif(os.path.exists("/dev/kfd"),
                    reason="build check: runs where the library is built, not on a GPU host "
                           "(no child processes next to an initialised GPU)")
def test_library_assembly_is_clean():
    r = subprocess.run(["make", "-C", PKG, "check"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
