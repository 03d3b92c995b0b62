"""The look through the assembly of kernels that name accumulation registers: what
the build ends for (CPU). The assembly is written here, with each mistake planted."""

import importlib.util
import os

import pytest

import deepspeed_amd

_PATH = os.path.join(os.path.dirname(deepspeed_amd.__file__), "ops",
                     "named_registers.py")
_spec = importlib.util.spec_from_file_location("named_registers", _PATH)
look = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(look)


def _assembly(body, scratch=0, spilled=0):
    text = ["wide:                  ; @wide", "; %bb.0:"]
    for line in body.strip().split("\n"):
        line = line.strip()
        if line.startswith("own "):
            text += ["\t;;#ASMSTART", "\t" + line[4:], "\t;;#ASMEND"]
        elif line.startswith("."):
            text.append(line)
        else:
            text.append("\t" + line)
    text += [".Lfunc_end0:", "\t.amdhsa_kernel wide",
             "\t\t.amdhsa_private_segment_fixed_size %d" % scratch,
             "\t.end_amdhsa_kernel", "    .name:           wide",
             "    .vgpr_spill_count: %d" % spilled]
    return "\n".join(text)


GOOD = """
    v_mov_b32_e32 v5, v6
    v_readfirstlane_b32 s4, v9
    s_nop 2
    .LBB0_1:
    own s_add_u32 m0, s9, 4
    own v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
    own buffer_load_dwordx4 v8, s[4:7], s8 offen lds
    ds_read_b128 v[0:3], v10 ; a comment on a[0:3] and m0
    s_cbranch_scc1 .LBB0_1
    own v_accvgpr_read_b32 v0, a[0:0]
    s_endpgm
"""


def test_nothing_to_find():
    assert look.faults(_assembly(GOOD)) == ([], 1)
    # kernels that name none are not looked at
    assert look.faults(_assembly("v_accvgpr_write_b32 a0, v0\ns_endpgm", 20)) == \
        ([], 0)


@pytest.mark.parametrize("now,then,what", [
    # taken by the compiler, alone and in a row
    ("ds_read_b128 v[0:3], v10", "v_accvgpr_write_b32 a255, v0", "outside"),
    ("ds_read_b128 v[0:3], v10", "ds_read_b128 a[252:255], v10", "outside"),
    ("ds_read_b128 v[0:3], v10", "s_mov_b32 m0, s2", "outside"),
    # written right before a product, by a pair as well
    ("own s_add_u32 m0, s9, 4", "v_mov_b32_e32 v7, v6\nown s_add_u32 m0, s9, 4",
     "right after"),
    ("own s_add_u32 m0, s9, 4", "v_permlane16_swap_b32 v20, v2\ns_nop 0",
     "right after"),
    ("own s_add_u32 m0, s9, 4", "v_mov_b32_e32 v7, v6\ns_nop 1", None),
    # and around the loop, where the branch and the addition lie between
    ("s_cbranch_scc1", "v_add_u32_e32 v3, 1, v3\ns_cbranch_scc1", None),
    # a vector instruction's scalar too close to a load's
    ("s_nop 2", "s_nop 1", "right after"),
])
def test_mistakes_are_found(now, then, what):
    assert now in GOOD
    bad, kernels = look.faults(_assembly(GOOD.replace(now, then)))
    assert kernels == 1
    assert bad if what else not bad
    assert all(what in b for b in bad)


def test_around_a_loop():
    text = GOOD.replace("s_cbranch_scc1", "v_add_u32_e32 v3, 1, v3\ns_cbranch_scc1")
    bad, _ = look.faults(_assembly(text.replace("own s_add_u32 m0, s9, 4", "s_nop 0")))
    assert bad == []
    bad, _ = look.faults(_assembly(text.replace("own s_add_u32 m0, s9, 4", "")))
    assert any("right after v_add_u32" in b for b in bad)


def test_memory_is_found():
    assert look.faults(_assembly(GOOD, scratch=20))[0] == ["wide: scratch memory"]
    assert look.faults(_assembly(GOOD, spilled=1))[0] == \
        ["wide: vector registers spilled"]
    # a compiler that no longer says so
    text = _assembly(GOOD).replace("private_segment", "other")
    assert look.faults(text)[0] == ["wide: scratch memory"]


class _Given:
    def __init__(self, text):
        self._text = text

    def text(self):
        return self._text


def test_the_build_ends():
    look.check(_Given(_assembly(GOOD)), "source", 1)
    with pytest.raises(RuntimeError, match="1 kernels name registers, not 2"):
        look.check(_Given(_assembly(GOOD)), "source", 2)
    with pytest.raises(RuntimeError, match="scratch"):
        look.check(_Given(_assembly(GOOD, scratch=4)), "source", 1)
