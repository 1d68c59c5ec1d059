"""The inline asm of the LM head kernels keeps gfx950's software wait states
(the generated assembly of each source, checked by tests/mfma_hazards.py)."""
from __future__ import annotations

import re

import pytest

import isa_listing
from mfma_hazards import hazards, hazards_of_kernel

MFMA = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"
COPY = "buffer_load_dwordx4 v9, s[4:7], s8 offen lds"

CASES = [  # (wait states needed, writer, reader)
    (2, "v_add_u32_e32 v5, v10, v11", MFMA),
    (2, "v_accvgpr_write_b32 a2, v10", MFMA),
    (2, "v_permlane32_swap_b32 v10, v2", MFMA),
    (5, "v_readlane_b32 s6, v10, 3", COPY),
    (5, "v_readfirstlane_b32 s8, v10", COPY),
    (5, "v_mad_u64_u32 v[10:11], s[6:7], v12, v13, v[14:15]", COPY),
    (1, "s_mov_b32 m0, s2", COPY),
    (1, "s_add_i32 m0, s2, 0x1000", COPY),
    (11, MFMA, "v_accvgpr_read_b32 v10, a3"),
    (11, MFMA, "v_accvgpr_write_b32 a3, v10"),
    (11, MFMA, "global_store_dwordx4 v[12:13], a[0:3], off"),
    (2, MFMA, MFMA),
]


@pytest.mark.parametrize("states,writer,reader", CASES)
def test_detector_counts_wait_states(states, writer, reader):
    for n in range(states + 1):
        body = ["; %bb.0:", "\t" + writer] + ["\ts_add_u32 s40, s41, s42"] * n
        found = hazards_of_kernel(body + ["\t" + reader, "\ts_endpgm"])
        assert bool(found) == (n < states), (n, found)
    if states > 1:
        body = ["; %bb.0:", "\t" + writer, f"\ts_nop {states - 1}", "\t" + reader, "\ts_endpgm"]
        assert not hazards_of_kernel(body)


def test_detector_follows_branches_and_other_registers():
    loop = ["; %bb.0:", "\tv_mov_b32_e32 v20, 0", ".LBB0_1:", "\t" + MFMA,
            "\tv_add_u32_e32 v1, v10, v11", "\ts_cbranch_scc0 .LBB0_1", "; %bb.2:", "\ts_endpgm"]
    assert [f[0] for f in hazards_of_kernel(loop)] == [MFMA]
    loop[4] = "\tv_add_u32_e32 v8, v10, v11"
    assert hazards_of_kernel(loop) == []
    # the SGPR written again by the scalar unit
    again = ["; %bb.0:", "\tv_readlane_b32 s6, v10, 3", "\ts_mov_b32 s6, s3", "\t" + COPY]
    assert hazards_of_kernel(again) == []


@pytest.mark.skipif(not isa_listing.available(), reason="hipcc not available")
@pytest.mark.parametrize("source", ["klp_lmhead.hip", "klp_head_gemm.hip"])
def test_kernels_have_wait_states(source):
    listing = isa_listing.listing(source)
    assert len(re.findall(r"^\s+v_mfma_", listing, re.M)) > 0
    found = hazards(listing)
    assert not found, {k: v[:2] for k, v in found.items()}


@pytest.mark.skipif(not isa_listing.available(), reason="hipcc not available")
def test_asm_copies_are_the_only_use_of_m0():
    """The copies written in asm cannot name m0 as clobbered: nothing else in
    their kernels may use it."""
    listing = isa_listing.listing("klp_head_gemm.hip")
    blocks = [b for b in re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", listing, re.S)
              if "buffer_load_dwordx4" in b]
    assert blocks and all("s_mov_b32 m0" in b for b in blocks)
    uses = [s for s in listing.splitlines() if re.search(r"\bm0\b", s.split(";")[0])]
    assert len(uses) == len(blocks)
