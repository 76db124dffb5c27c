"""check_waits.py, which every build runs over the compiled prefill kernels: it
passes code whose barriers come after a wait that covers the LDS loads, and
finds the ways in which a compiler could break that.
"""

import importlib.util
import os

import pytest

PATH = os.path.join(os.path.dirname(__file__), "..", "molla_amd", "csrc", "check_waits.py")
ASM = os.path.join(os.path.dirname(PATH), "_obj", "prefill-hip-amdgcn-amd-amdhsa-gfx950.s")
spec = importlib.util.spec_from_file_location("check_waits", PATH)
check_waits = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_waits)

GOOD = """
.LBB0_1:                                ; =>This Inner Loop Header
	s_mov_b32 m0, s35
	global_load_lds_dwordx4 v46, s[8:9]
	s_mov_b32 m0, s36
	global_load_lds_dwordx4 v46, s[8:9]
	global_load_dwordx4 v[0:3], v[4:5], off
	global_load_dword v6, v[4:5], off offset:16
	; sched_barrier mask(0x00000000)
	ds_read_b128 v[8:11], v7
	s_waitcnt lgkmcnt(0)
	s_waitcnt vmcnt(2)
	s_barrier
	s_cbranch_scc1 .LBB0_1
	s_endpgm
"""
LOAD = "	global_load_dword v6, v[4:5], off offset:16\n"


def run(text):
    return check_waits.check(text.splitlines())


def test_covered_loads_pass():
    assert run(GOOD) == (2, [])


@pytest.mark.parametrize("name,text", [
    ("two loads merged into one", GOOD.replace(LOAD, "")),
    ("a load moved ahead of the transfer", GOOD.replace(LOAD, "").replace("	s_mov_b32 m0, s35\n", LOAD + "	s_mov_b32 m0, s35\n")),
    ("a load moved behind the wait", GOOD.replace(LOAD, "").replace("	s_barrier\n", LOAD + "	s_barrier\n")),
    ("a store is no load", GOOD.replace(LOAD, "	global_store_dword v[4:5], v6, off\n")),
    ("m0 read by other code", GOOD.replace("	ds_read", "	s_add_u32 s3, m0, s4\n	ds_read")),
    ("a load on the m0 of another", GOOD.replace("	s_mov_b32 m0, s36\n", "")),
    ("the wait is gone", GOOD.replace("	s_waitcnt vmcnt(2)\n", "")),
    ("a branch round the wait", GOOD.replace("	s_waitcnt vmcnt(2)\n", "	s_cbranch_execz .LBB0_2\n	s_waitcnt vmcnt(2)\n.LBB0_2:\n")),
])
def test_broken_order_is_found(name, text):
    seen, bad = run(text)
    assert seen == 2 and bad, name


def test_the_built_kernels():
    if not os.path.exists(ASM):
        pytest.skip("the library was not built here")
    with open(ASM) as f:
        seen, bad = run(f.read())
    # 24 kernels of eight kinds, each with four stages and a first one
    assert seen >= 24 * 5 and not bad
