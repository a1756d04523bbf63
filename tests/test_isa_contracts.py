"""What the hand-written assembly in the kernels relies on, checked on the compiler's output.

The compiler inserts the wait states gfx90a-and-later hardware needs between dependent
instructions, but only around instructions it can see -- not around inline assembly:
  * a vector-memory instruction must not read an SGPR that a VALU instruction (v_readfirstlane,
    v_cmp with a scalar destination, ...) wrote within the five instructions before it;
  * a VALU instruction must not read an SGPR that a VALU instruction wrote within the two before it.
`dma_load` (kernels_gemm.hip: s_mov m0 / s_nop / global_load_lds) relies on its scalar operands
coming from scalar instructions; `set_lane2` (kernels_gate.hip) carries its own s_nop.  This test
compiles both files to gfx950 assembly (no GPU needed) and checks every assembly block along every
path that reaches it (fall-through, branches from other blocks, loop back-edges).

The GEMM's k loops also wait for their global->LDS loads with hand-counted `s_waitcnt vmcnt(n)`:
that count is right only while those loads are the only vector-memory instructions a wave issues
between the first and the last of them, which the second test checks for every instantiation."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cuspamm_amd", "csrc")


def _isa(src, tmp_path):
    from cuspamm_amd import build
    out = os.path.join(str(tmp_path), src.replace(".hip", ".s"))
    cmd = [build.HIPCC] + [f for f in build.CFLAGS if f != "-Wall"] + build.EXTRA_FLAGS.get(src, []) + ["-S", "--cuda-device-only",
                                                                                                     os.path.join(CSRC, src), "-o", out]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    return open(out).read()


def _sgprs(token):
    """SGPR numbers named by one operand: s5 -> {5}, s[10:11] -> {10, 11}, vcc -> {'vcc'}."""
    token = token.strip().rstrip(",")
    m = re.fullmatch(r"s(\d+)", token)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", token)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    if token in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc"}
    return set()


def _instructions(text):
    """(mnemonic, operands, inside an inline-assembly block) per instruction line, in order; a label
    line gives ("label:", [name], False)."""
    out, in_asm = [], False
    for line in text.splitlines():
        s = line.strip()
        if s.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if s.startswith(";;#ASMEND"):
            in_asm = False
            continue
        if not s or s.startswith((";", "/")):
            continue
        s = s.split(";")[0].strip()
        if not s:
            continue
        m = re.fullmatch(r"([.\w$]+):", s)
        if m:
            out.append(("label:", [m.group(1)], False))
            continue
        if s.startswith("."):
            continue
        parts = s.split(None, 1)
        ops = [o.strip() for o in parts[1].split(",")] if len(parts) > 1 else []
        out.append((parts[0], ops, in_asm))
    return out


def _valu_written_sgprs(mnemonic, ops):
    """SGPRs a VALU instruction writes (scalar destination of a v_ instruction)."""
    if not mnemonic.startswith("v_") or not ops:
        return set()
    written = _sgprs(ops[0])
    if mnemonic.startswith(("v_cmp", "v_cmpx")) and mnemonic.endswith("_e32"):
        written |= {"vcc"}
    if re.match(r"v_(add|sub|subrev)_co_", mnemonic) and len(ops) > 1:
        written |= _sgprs(ops[1])
    return written


def _wait_states(mnemonic, ops):
    if mnemonic == "s_nop" and ops:
        return int(ops[0], 0) + 1
    return 1


def _hazards(ins, reader, need):
    """Every (reader index, offending instruction index) where an inline-assembly `reader` reads an SGPR
    that a VALU instruction wrote fewer than `need` wait states earlier, along ANY path: at a label
    the walk goes on into the fall-through predecessor and into every block that branches there
    (loop back-edges included)."""
    labels = {ops[0]: i for i, (mn, ops, _) in enumerate(ins) if mn == "label:"}
    branches = {}
    for i, (mn, ops, _) in enumerate(ins):
        if mn.startswith(("s_branch", "s_cbranch")) and ops and ops[0] in labels:
            branches.setdefault(ops[0], []).append(i)
    found, checked = [], 0

    def walk(j, states, read, origin, seen):
        while j >= 0 and states < need:
            pmn, pops, _ = ins[j]
            if pmn == "label:":
                for b in branches.get(pops[0], []):
                    if (b, states) not in seen:
                        seen.add((b, states))
                        walk(b, states, read, origin, seen)         # the branch itself is one wait state, counted there
                if j > 0 and ins[j - 1][0] == "s_branch":
                    return                                          # no fall-through into this label
                j -= 1
                continue
            if _valu_written_sgprs(pmn, pops) & read:
                found.append((origin, j))
            states += _wait_states(pmn, pops)
            j -= 1

    for i, (mn, ops, in_asm) in enumerate(ins):
        if not in_asm or mn != reader:
            continue
        checked += 1
        read = set()
        for o in ops:
            read |= _sgprs(o.split()[0]) if o else set()
        walk(i - 1, 0, read, i, set())
    return found, checked


@pytest.mark.parametrize("src,reader,need", [("kernels_gemm.hip", "global_load_lds_dwordx4", 5),
                                             ("kernels_gate.hip", "v_writelane_b32", 2)])
def test_assembly_blocks_keep_their_distance_from_valu_written_sgprs(tmp_path, src, reader, need):
    ins = _instructions(_isa(src, tmp_path))
    found, checked = _hazards(ins, reader, need)
    for origin, j in found:
        mn, ops, _ = ins[origin]
        pmn, pops, _ = ins[j]
        raise AssertionError("%s: %s %s reads an SGPR written too shortly before by %s %s" % (
            src, mn, ", ".join(ops), pmn, ", ".join(pops)))
    assert checked > 20, "no %s found inside assembly blocks of %s" % (reader, src)


FIXTURE_STRAIGHT = """
k:
    v_readfirstlane_b32 s4, v1
    s_mov_b32 s5, 0
    s_nop 0
    ;;#ASMSTART
    s_mov_b32 m0, s9
    s_nop 0
    global_load_lds_dwordx4 v2, s[4:5] offset:0
    ;;#ASMEND
    s_endpgm
"""
FIXTURE_BACK_EDGE = """
k:
    s_mov_b32 s4, 0
    s_mov_b32 s5, 0
    s_nop 4
.LBB0_1:
    ;;#ASMSTART
    s_mov_b32 m0, s9
    s_nop 0
    global_load_lds_dwordx4 v2, s[4:5] offset:0
    ;;#ASMEND
    s_add_u32 s8, s8, 1
    v_readfirstlane_b32 s4, v1
    s_cmp_lt_u32 s8, s10
    s_cbranch_scc1 .LBB0_1
    s_endpgm
"""
FIXTURE_OTHER_PREDECESSOR = """
k:
    s_cbranch_scc1 .LBB0_2
    v_readfirstlane_b32 s4, v1
    s_branch .LBB0_3
.LBB0_2:
    s_mov_b32 s4, 0
    s_nop 4
.LBB0_3:
    ;;#ASMSTART
    s_mov_b32 m0, s9
    s_nop 0
    global_load_lds_dwordx4 v2, s[4:5] offset:0
    ;;#ASMEND
    s_endpgm
"""
FIXTURE_CLEAN_LOOP = """
k:
    v_readfirstlane_b32 s4, v1
    s_nop 4
.LBB0_1:
    ;;#ASMSTART
    s_mov_b32 m0, s9
    s_nop 0
    global_load_lds_dwordx4 v2, s[4:5] offset:0
    ;;#ASMEND
    s_add_u32 s4, s4, 64
    s_addc_u32 s5, s5, 0
    s_cmp_lt_u32 s4, s10
    s_cbranch_scc1 .LBB0_1
    s_endpgm
"""


def test_hazard_checker_sees_hazards_across_branches():
    # the checker itself: a hazard in straight-line code, over a loop back-edge and from a second
    # predecessor block must each be reported; a loop whose address is advanced by scalar
    # instructions only must pass
    for text, want in ((FIXTURE_STRAIGHT, 1), (FIXTURE_BACK_EDGE, 1), (FIXTURE_OTHER_PREDECESSOR, 1), (FIXTURE_CLEAN_LOOP, 0)):
        found, checked = _hazards(_instructions(text), "global_load_lds_dwordx4", 5)
        assert checked == 1 and len(found) == want, (text, found)


def test_gemm_k_loops_issue_no_other_vector_memory_instruction(tmp_path):
    text = _isa("kernels_gemm.hip", tmp_path)
    kernels = re.findall(r"^(_ZN5spamm(?:6k_gemm|10k_gemm_w64)ILi\d+ELi\d+(?:ELi\d+|ELb[01])?EEE\w+):[^\n]*\n(.*?)s_endpgm", text, flags=re.S | re.M)
    # whole macro tiles by four waves: tiles 32 / 64 / 128 x ring depths 3 / 4 / 5, and the three tiles by
    # workgroups that stay (ELb1E); waves of 64 x 128 (half macro tiles, whole macro tiles by eight waves):
    # the three tiles each
    assert len([n for n, _ in kernels if "k_gemm_w64" not in n and "ELb0E" in n]) == 9
    assert len([n for n, _ in kernels if "k_gemm_w64" not in n and "ELb1E" in n]) == 3
    assert len([n for n, _ in kernels if "k_gemm_w64" in n]) == 6
    for name, body in kernels:
        mns = [mn for mn, _, _ in _instructions(body)]
        dma = [i for i, mn in enumerate(mns) if mn == "global_load_lds_dwordx4"]
        assert len(dma) >= 12, name
        other = [mn for mn in mns[dma[0]:dma[-1] + 1]
                 if mn.startswith(("global_", "flat_", "buffer_", "scratch_")) and mn != "global_load_lds_dwordx4"]
        assert not other, "%s: %s between the first and the last global->LDS load" % (name, sorted(set(other)))
        # and C is stored only after the loops have drained the ring
        stores = [i for i, mn in enumerate(mns) if mn.startswith("global_store")]
        assert stores and min(i for i in stores if i > dma[0]) > dma[-1], name
        # workgroups that stay draw their tickets with a returning atomic: it must be issued before an
        # item's first global->LDS load (then it is older than every load the counts speak of); the
        # stores of the previous item's C are older than the next item's loads in the same way
        # (a third one sits in the loop over the items with nothing kept, after the last load)
        atomics = [i for i, mn in enumerate(mns) if mn.startswith("global_atomic")]
        if "ELb1E" in name:
            assert len([i for i in atomics if i < dma[0]]) == 2 and len([i for i in atomics if i > dma[-1]]) == 1, name
            assert not any(mn.startswith("scratch_") for mn in mns), name
        else:
            assert not atomics, name


def test_small_output_kernel_keeps_the_same_contracts(tmp_path):
    # kernels_small.hip: three tile sizes x units of 128 and 64, the same assembly blocks and hand-counted waits
    text = _isa("kernels_small.hip", tmp_path)
    ins = _instructions(text)
    for reader in ("global_load_lds_dwordx4", "global_store_dword"):
        found, checked = _hazards(ins, reader, 5)
        assert not found and checked > 20, (reader, [ins[i] for pair in found for i in pair])
    found, checked = _hazards(_instructions(_isa("kernels_gemm.hip", tmp_path)), "global_store_dword", 5)
    assert not found and checked > 20
    kernels = re.findall(r"^(_ZN5spamm7k_smallILi\d+ELi\d+EEE\w+):[^\n]*\n(.*?)s_endpgm", text, flags=re.S | re.M)
    assert len(kernels) == 6
    for name, body in kernels:
        mns = [mn for mn, _, _ in _instructions(body)]
        dma = [i for i, mn in enumerate(mns) if mn == "global_load_lds_dwordx4"]
        assert len(dma) >= 12, name
        other = [mn for mn in mns[dma[0]:dma[-1] + 1]
                 if mn.startswith(("global_", "flat_", "buffer_", "scratch_")) and mn != "global_load_lds_dwordx4"]
        assert not other, "%s: %s between the first and the last global->LDS load" % (name, sorted(set(other)))
        assert not any(mn.startswith("scratch_") for mn in mns), name


def test_three_small_units_per_cu_keep_the_same_contracts(tmp_path):
    # the ring of three: no other vector-memory instruction between its loads, no scratch
    text = _isa("kernels_small.hip", tmp_path)
    kernels = re.findall(r"^(_ZN5spamm13k_small_threeILi\d+EEE\w+):[^\n]*\n(.*?)s_endpgm", text, flags=re.S | re.M)
    assert len(kernels) == 3
    for name, body in kernels:
        mns = [mn for mn, _, _ in _instructions(body)]
        dma = [i for i, mn in enumerate(mns) if mn == "global_load_lds_dwordx4"]
        assert len(dma) >= 12, name
        memory = {mn for mn in mns[dma[0]:dma[-1] + 1] if mn.startswith(("global_", "flat_", "buffer_", "scratch_"))}
        assert memory == {"global_load_lds_dwordx4"} and not any(mn.startswith("scratch_") for mn in mns), name


def test_small_output_kernels_read_their_arguments_from_two_lines(tmp_path):
    # a later line of arguments would be fetched when M, N and C are needed, in the middle of the kernel's chain
    text = _isa("kernels_small.hip", tmp_path)
    kernels = re.findall(r"^(_ZN5spamm(?:7k_small|13k_small_three)I\w+):[^\n]*\n(.*?)s_endpgm", text, flags=re.S | re.M)
    assert len(kernels) == 9
    for name, body in kernels:
        loads = re.findall(r"s_load_dword(?:x(\d+))?\s+\S+, s\[\d+:\d+\], (0x[0-9a-f]+)", body)
        assert loads and max(int(at, 16) + 4 * int(n or 1) for n, at in loads) <= 128, (name, loads)


def test_small_output_kernels_read_lds_soon_behind_a_sync(tmp_path):
    # gate, list, prologue, then two full and two partial stages a turn: a full stage has an entry's read, its address and
    # its own reads' in front of them
    text = _isa("kernels_small.hip", tmp_path)
    kernels = re.findall(r"^(_ZN5spamm(?:7k_small|13k_small_three)I\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, flags=re.S | re.M)
    assert len(kernels) == 9
    for name, body in kernels:
        lines = [ln for ln in (re.sub(r";.*", "", ln).strip() for ln in body.splitlines()) if ln and not ln.startswith(".")]
        syncs = [i for i, ln in enumerate(lines) if ln.startswith("s_barrier")]
        assert len(syncs) == 7, name
        for at in syncs[3:5]:
            reads = next(i for i in range(at, len(lines)) if lines[i].startswith("ds_read_b128"))
            assert reads - at <= 8, (name, reads - at)


def test_results_are_published_when_the_workspace_is_at_rest(tmp_path):
    """The host goes on when it sees a result's sequence number and may use the workspace at once, from another stream:
    behind a publishing kernel's last barrier no wave stores anything but the result itself (to host memory, in system
    scope: sc0 sc1), and in the kernel whose waves all clear counters, every wave has waited for its stores before it."""
    publishing = [("kernels_tau.hip", r"_ZN5spamm10k_tau_histILi2E\w+", 1), ("kernels_tools.hip", r"_ZN5spamm13k_error_denseILi\w+", 3),
                  ("kernels_tools.hip", r"_ZN5spamm15k_dropped_bound\w+", 1), ("kernels_tools.hip", r"_ZN5spamm13k_error_limbs\w+", 1)]
    for src, name, count in publishing:
        kernels = re.findall(r"^(%s):[^\n]*\n(.*?)^\.Lfunc_end" % name, _isa(src, tmp_path), flags=re.S | re.M)
        assert len(kernels) == count, src
        for kernel, body in kernels:
            lines = [ln.strip() for ln in body.splitlines()]
            last = max(i for i, ln in enumerate(lines) if ln.startswith("s_barrier"))
            stores = [ln for ln in lines[last:] if re.match(r"(global|flat|buffer|scratch)_(store|atomic)", ln)]
            assert stores and all(ln.endswith("sc0 sc1") for ln in stores), (kernel, stores)
            if "k_tau_hist" in kernel:
                block = []
                for ln in reversed(lines[:last]):
                    if ln.startswith("s_barrier"):
                        break
                    block.append(ln)
                waits = [i for i, ln in enumerate(block) if re.match(r"s_waitcnt.*vmcnt\(0\)", ln)]
                clears = [i for i, ln in enumerate(block) if ln.startswith("global_store")]
                assert clears and waits and waits[0] < clears[0], kernel        # (reversed: the last wait comes after the last store)
                assert not any(ln.startswith((".LBB", "s_cbranch", "s_branch")) for ln in block[:waits[0]]), kernel


def test_bisection_state_is_stored_past_the_cache(tmp_path):
    """The bisection's state is read by the next call, on whatever stream, as soon as the host has seen a result: no
    kernel of it stores to global memory but past its XCD's cache (sc1)."""
    text = _isa("kernels_tau.hip", tmp_path)
    for name in ("k_tau_count", "k_tau_tree"):
        kernels = re.findall(r"^(_ZN5spamm\d+%s\w+):[^\n]*\n(.*?)^\.Lfunc_end" % name, text, flags=re.S | re.M)
        assert len(kernels) == 1
        stores = [ln.strip() for ln in kernels[0][1].splitlines() if re.match(r"\s*(global|flat|buffer|scratch)_store", ln)]
        assert stores and all("sc1" in ln for ln in stores), (name, stores)


def test_bisection_publishes_when_its_workspace_is_at_rest(tmp_path):
    """The same for the bisection, which publishes from the launch that ends it: behind the last barrier one thread stores the
    state, then the result, waits, and stores the sequence number; and every wave of the tree, all of which clear leaves, has
    waited for its stores before a barrier in between."""
    text = _isa("kernels_tau.hip", tmp_path)
    for name, waits in (("k_tau_count", 1 + 2), ("k_tau_tree", 1 + 1 + 1)):     # last_workgroup, the leaves, publish_result (two calls)
        (body,) = re.findall(r"^_ZN5spamm\d+%s\w+:[^\n]*\n(.*?)^\.Lfunc_end" % name, text, flags=re.S | re.M)
        lines = [ln.strip() for ln in body.splitlines()]
        asm = [i for i, ln in enumerate(lines) if re.match(r"s_waitcnt vmcnt\(0\)$", ln) and lines[i - 1].startswith(";;#ASMSTART")]
        assert len(asm) == waits, (name, asm)
        last = max(i for i, ln in enumerate(lines) if ln.startswith("s_barrier"))
        assert asm[-1] > last
        end = [i for i in range(last, len(lines)) if re.match(r"(global|flat|buffer|scratch)_(store|atomic)", lines[i])]
        results = [i for i in end if "sc0 sc1" in lines[i]]
        assert all("sc1" in lines[i] for i in end) and results[-1] == end[-1] and asm[-1] == max(i for i in asm if i < end[-1])
        assert not [i for i in end[:-1] if i > asm[-1]], name                   # the sequence number alone comes behind the wait
        if name == "k_tau_tree":
            rest = lines[asm[1] + 1:]
            barrier = next(i for i, ln in enumerate(rest) if ln.startswith("s_barrier"))
            assert not any(re.match(r"\.LBB|s_cbranch|s_branch|global_|flat_", ln) for ln in rest[:barrier]) and asm[1] + 1 + barrier < last
            clears = [i for i, ln in enumerate(lines) if ln.startswith("global_store") and asm[0] < i < last]
            assert len(clears) >= 4, clears


def test_integer_product_keeps_the_same_distance(tmp_path):
    """kernels_tools.hip: the planes' addresses come through v_readlane, and the global->LDS loads take what scalar instructions
    make of it; the accumulators of seven orders stay in registers."""
    text = _isa("kernels_tools.hip", tmp_path)
    found, checked = _hazards(_instructions(text), "global_load_lds_dwordx4", 5)
    assert not found and checked > 20, found
    ((_, body),) = re.findall(r"^(_ZN5spamm13k_error_limbs\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, flags=re.S | re.M)
    assert not any(mn.startswith("scratch_") for mn, _, _ in _instructions(body))


def test_single_pass_of_two_groups_leaves_room_for_a_third_workgroup(tmp_path):
    """kernels_normmap.hip: the fp32 pass of A = B with two 8-row groups per lane lives from three workgroups per CU, which 42 KiB of
    LDS and up to 168 registers allow; nothing is spilled for it."""
    text = _isa("kernels_normmap.hip", tmp_path)
    found = re.findall(r"\.name:\s+_ZN5spamm9k_normmapILi64ELi2ELi256ELb0ELi1ELi4E\w*.*?\.vgpr_count:\s+(\d+)\s+\.vgpr_spill_count:\s+(\d+)", text, flags=re.S)
    assert found and all(int(n) <= 168 and int(spilled) == 0 for n, spilled in found), found


def test_lds_written_16_bytes_at_a_time_is_declared_for_it():
    """The compiler gives larger arrays 16 bytes by itself, which nothing promises: what is written or read by vectors of 16 bytes
    says so where it is declared."""
    seen = 0
    for src in sorted(os.listdir(CSRC)):
        if not src.endswith((".hip", ".h")):
            continue
        text = open(os.path.join(CSRC, src)).read()
        wide = set(re.findall(r"reinterpret_cast<(?:const )?(?:u32x4n?|i32x4|f32x4|uint4|half8t) \*>\((s_\w+)", text))
        for decl in re.findall(r"^\s*__shared__ ([^;]*);", text, flags=re.M):
            names = set(re.findall(r"(s_\w+)\[", decl)) & wide
            seen += len(names)
            assert not names or "aligned(16)" in decl, (src, decl)
    assert seen >= 3


def test_wide_stores_written_out_keep_their_data(tmp_path):
    """A vector instruction may not write the registers of a store of more than 64 bits within two wait states of it, which the
    compiler sees to around stores of its own: the ones written out carry the wait states."""
    for src, least in (("kernels_normmap.hip", 21), ("kernels_tools.hip", 4)):
        ins = _instructions(_isa(src, tmp_path))
        wide = [i for i, (mn, _, in_asm) in enumerate(ins) if in_asm and mn in ("global_store_dwordx4", "global_store_dwordx3")]
        assert len(wide) >= least, src
        for i in wide:
            mn, ops, _ = ins[i + 1]
            assert mn == "s_nop" and int(ops[0], 0) >= 1, ins[i:i + 2]


def test_one_word_kernels_keep_the_same_contracts(tmp_path):
    """The one-launch kernels whose list is a register: their buffer->LDS loads keep their distance from VALU-written SGPRs and are the only
    vector-memory instructions between the first and the last of them, nothing is spilled, and the arguments lie in two lines."""
    text = _isa("kernels_small.hip", tmp_path)
    found, checked = _hazards(_instructions(text), "buffer_load_dwordx4", 5)
    assert not found and checked > 60, found
    kernels = re.findall(r"^(_ZN5spamm(?:7k_small|13k_small_three)ENS_8WordArgs\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, flags=re.S | re.M)
    assert len(kernels) == 9
    for name, body in kernels:
        ins = _instructions(body)
        dma = [i for i, (mn, _, in_asm) in enumerate(ins) if in_asm and mn == "buffer_load_dwordx4"]
        assert len(dma) >= 12, name
        other = [mn for i, (mn, _, _) in enumerate(ins) if dma[0] <= i <= dma[-1] and i not in dma and mn.startswith(("global_", "flat_", "buffer_", "scratch_"))]
        assert not other and not any(mn.startswith("scratch_") for mn, _, _ in ins), (name, other)
        loads = re.findall(r"s_load_dword(?:x(\d+))?\s+\S+, s\[\d+:\d+\], (0x[0-9a-f]+)", body)
        assert loads and max(int(at, 16) + 4 * int(n or 1) for n, at in loads) <= 128, (name, loads)


@pytest.mark.parametrize("src", ["kernels_gate.hip", "kernels_normmap.hip"])
def test_offsets_that_no_buffer_holds_stay_within_their_type(src, tmp_path):
    """A lane with nothing to load gets an offset beyond its buffer.  Signed arithmetic on it that leaves 31 bits may be taken by the compiler
    as never happening, and with it the offset: looked for in the optimised intermediate code, where a value that is one of two has a
    large constant among them and goes into a signed operation with another constant."""
    from cuspamm_amd import build
    out = os.path.join(str(tmp_path), "ir.ll")
    cmd = [build.HIPCC] + [f for f in build.CFLAGS if f != "-Wall"] + build.EXTRA_FLAGS.get(src, []) + ["-S", "-emit-llvm", "--cuda-device-only",
                                                                                                    os.path.join(CSRC, src), "-o", out]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    wrong, selects = [], 0
    operate = {"add": lambda x, y: x + y, "mul": lambda x, y: x * y, "shl": lambda x, y: x << y}
    for function in open(out).read().split("\ndefine ")[1:]:
        chosen = {}
        for name, rest in re.findall(r"(%\S+) = (?:select|phi) (.*)", function):
            large = [int(c) for c in re.findall(r"i32 (-?\d{9,})", rest) + re.findall(r"\[ (-?\d{9,}), ", rest)]
            if large:
                chosen[name] = large
        selects += len(chosen)
        for op, name, c in re.findall(r"= (add|mul|shl) (?:nuw )?nsw i32 (%\S+), (-?\d+)", function):
            wrong += [(op, v, int(c)) for v in chosen.get(name, []) if not -2 ** 31 <= operate[op](v, int(c)) < 2 ** 31]
    assert selects and not wrong, wrong
