"""The check of the compiler's device listings (cardiacfoam_amd/listing.py) on short listings:
a register copied ahead of a join's mask restore is found where only that copy reaches a
read, and nothing else is."""
import pytest

from cardiacfoam_amd.listing import masked_reads

HEAD = """_Zkern:
; %bb.0:
\tv_mov_b32_e32 v0, 0
\tv_cmp_gt_i32_e32 vcc, 4, v1
\ts_mov_b32 s6, 8
"""
TAIL = """\ts_endpgm
.Lfunc_end0:
"""
# lanes that take the branch read a word; at the join v8 goes to a4
JOIN = """.LBB0_1:
{before}\ts_and_saveexec_b64 s[0:1], vcc
{branch}; %bb.2:
\tds_read_b32 v3, v0
{in_body}; %bb.3:
\tv_writelane_b32 v9, s6, 3
{at_join}\ts_or_b64 exec, exec, s[0:1]
{after}\ts_sub_i32 s6, s6, 1
\ts_cmp_lg_u32 s6, 0
\ts_cbranch_scc1 .LBB0_1
; %bb.4:
\tv_accvgpr_read_b32 v5, a4
"""
COPY = "\tv_accvgpr_write_b32 a4, v8\n"


def _run(tmp_path, text):
    p = tmp_path / "k.s"
    p.write_text(text)
    return masked_reads(str(p))


@pytest.mark.parametrize("where,found", [("at_join", True), ("after", False), ("in_body", False),
                                         ("before", False)])
def test_copy_at_a_join(tmp_path, where, found):
    """in_body: the branch's own lanes (a conditional value); after and before: all lanes."""
    parts = dict.fromkeys(("before", "branch", "in_body", "at_join", "after"), "")
    parts[where] = COPY
    hits = _run(tmp_path, HEAD + JOIN.format(**parts) + TAIL)
    assert bool(hits) == found
    if found:
        (reg, line, inst), = hits["_Zkern"]
        assert reg == "a4" and inst == "v_accvgpr_read_b32 v5, a4"


def test_copy_of_a_value_that_all_lanes_hold(tmp_path):
    """a write of the register under the full mask that reaches the same read: the copy can be
    the branch's side of a conditional value"""
    parts = dict.fromkeys(("before", "branch", "in_body", "at_join", "after"), "")
    parts["at_join"] = COPY
    text = HEAD + "\ts_cbranch_scc1 .LBB0_9\n" + JOIN.format(**parts) + "\ts_endpgm\n" + \
        ".LBB0_9:\n\tv_accvgpr_write_b32 a4, 0\n\tv_accvgpr_read_b32 v5, a4\n" + TAIL
    assert [h[0] for h in _run(tmp_path, text)["_Zkern"]] == ["a4"]      # the loop's read only
    merged = HEAD + "\tv_accvgpr_write_b32 a4, 0\n\ts_cbranch_scc1 .LBB0_9\n" + \
        JOIN.format(**parts).replace("; %bb.4:", ".LBB0_9:") + TAIL
    assert not _run(tmp_path, merged)


def test_body_that_ends_in_the_restore(tmp_path):
    """a branch over the body: what the body's block writes ahead of the restore is its own"""
    text = HEAD + """\ts_and_saveexec_b64 s[0:1], vcc
\ts_cbranch_execz .LBB0_2
.LBB0_1:
\tv_mov_b32_e32 v4, v8
\tds_write_b32 v0, v4
\ts_or_b64 exec, exec, s[0:1]
.LBB0_2:
\tv_mov_b32_e32 v6, v4
""" + TAIL
    assert not _run(tmp_path, text)


@pytest.mark.parametrize("copy,read", [("\tv_mov_b64_e32 v[20:21], v[8:9]\n", "v_add_f64 v[2:3], v[20:21], 1.0"),
                                       ("\tscratch_load_dwordx2 v[20:21], off, s32\n", "ds_write_b64 v0, v[20:21]")])
def test_other_copies(tmp_path, copy, read):
    parts = dict.fromkeys(("before", "branch", "in_body", "at_join", "after"), "")
    parts["at_join"] = copy
    text = HEAD + JOIN.format(**parts).replace("v_accvgpr_read_b32 v5, a4", read) + TAIL
    assert sorted(h[0] for h in _run(tmp_path, text)["_Zkern"]) == ["v20", "v21"]
