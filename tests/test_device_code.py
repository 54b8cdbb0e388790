"""What the built gfx950 code has to show that no run of it can: listings of libmlh.so's own kernels.  CPU only."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# Kernels whose workgroups publish partial results or phase outputs by bumping a counter.
COUNTING = ("k_gemm_tile", "k_gemm_skinny", "k_gemm_skinny16", "k_decode_persistent")


@pytest.fixture(scope="module")
def listing(pkg, tmp_path_factory):
    """{kernel: its instructions, in address order} of every device code object in the built library."""
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(os.path.join(pkg.LIB_DIR, "libmlh.so"), where / "libmlh.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=where, check=True, capture_output=True)
    out = {}
    for f in sorted(os.listdir(where)):
        if not f.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", f], cwd=where, check=True, capture_output=True, text=True).stdout
        code = None
        for line in text.splitlines():
            head = re.match(r"<(\S+)>:$|^[0-9a-f]+ <(\S+)>:$", line)
            if head:
                code = out.setdefault(head.group(1) or head.group(2), [])
            elif code is not None and line.strip():
                code.append(line.split("//")[0].strip())
    return out


def kernel_name(symbol):
    m = re.match(r"_Z(\d+)", symbol)
    return symbol[m.end():m.end() + int(m.group(1))] if m else symbol


def test_stores_have_landed_before_a_counter_says_so(listing):
    """A counter that tells other workgroups (of another XCD as a rule) that partial sums are in memory may go up only when every
    wave's stores have been acknowledged: in front of the barrier before the atomic, each wave waits for vmcnt(0) behind its last
    store.  A workgroup-scope release fence compiles to no such wait on this target."""
    seen, bad = {}, []
    for symbol, code in listing.items():
        name = kernel_name(symbol)
        if name not in COUNTING:
            continue
        for i, ins in enumerate(code):
            if not ins.startswith("global_atomic_add"):
                continue
            seen[name] = seen.get(name, 0) + 1
            b = next(k for k in range(i, -1, -1) if code[k].startswith("s_barrier"))
            for k in range(b - 1, -1, -1):
                op = code[k].split()[0]
                if op == "s_waitcnt" and re.search(r"vmcnt\(0\)", code[k]):
                    break
                if re.match(r"(global|flat|buffer|scratch)_(store|atomic)", op) or op.startswith(("s_cbranch", "s_branch", "s_setpc")):
                    bad.append((symbol, i, code[k]))
                    break
    assert set(seen) == set(COUNTING), seen
    assert not bad, f"{len(bad)} counters go up while stores may be on their way, the first: {bad[0]}"


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]|v(\d+)\b", operand)
    if not m:
        return set()
    return {int(m.group(3))} if m.group(3) else set(range(int(m.group(1)), int(m.group(2)) + 1))


def _overwrites(code, i, data, states=2):
    """The first vector instruction within `states` wait states behind code[i] that writes one of the registers `data` (s_nop N is N + 1 of them, any other
    instruction one; a taken branch takes longer than two)."""
    for ins in code[i + 1:]:
        if states <= 0 or ins.startswith(("s_branch", "s_setpc", "s_endpgm")):
            return None
        m = re.match(r"s_nop (\w+)", ins)
        states -= int(m.group(1), 0) + 1 if m else 1
        if ins.startswith("v_"):
            operands = ins.split(None, 1)[1].split(",")
            written = operands[:2] if "swap" in ins.split()[0] else operands[:1]
            if any(_registers(o.strip()) & data for o in written):
                return ins
    return None


def test_no_wide_stores_data_is_overwritten_while_it_is_read(listing):
    """A store of 12 or 16 bytes reads its data after it has been issued.  The compiler keeps two wait states between it and a write of
    those registers except where a buffer store has a scalar offset, and there lanes have stored the overwritten value."""
    stores, bad = 0, []
    for symbol, code in listing.items():
        for i, ins in enumerate(code):
            m = re.match(r"(buffer|global|flat|scratch)_store_dwordx[34] (.*)", ins)
            if not m:
                continue
            stores += 1
            operands = [o.strip() for o in m.group(2).split(",")]
            after = _overwrites(code, i, _registers(operands[0 if m.group(1) == "buffer" else 1]))
            if after:
                bad.append((symbol, ins, after))
    assert stores > 100
    assert not bad, f"{len(bad)} stores, the first: {bad[0]}"


def test_the_wait_states_behind_a_store():
    """What the check above counts: the instruction behind the next one, not what two or an s_nop of two wait states keep away, and both results of a swap."""
    data = _registers("v[4:7]")
    assert _overwrites(["store", "s_nop 0", "v_add_f32_e32 v5, v1, v2"], 0, data)
    assert _overwrites(["store", "v_mov_b32_e32 v1, v4", "v_add_f32_e32 v7, v1, v2"], 0, data)
    assert _overwrites(["store", "v_permlane16_swap_b32_e32 v1, v6"], 0, data)
    assert not _overwrites(["store", "s_branch 65115", "v_add_f32_e32 v5, v1, v2"], 0, data)
    assert not _overwrites(["store", "s_nop 1", "v_add_f32_e32 v5, v1, v2"], 0, data)
    assert not _overwrites(["store", "v_mov_b32_e32 v1, v4", "v_mov_b32_e32 v8, v4", "v_add_f32_e32 v7, v1, v2"], 0, data)


def test_every_built_form_of_the_decode_of_several_sequences_is_reached(listing):
    """fp32 weights with heads of 64, bf16 with 64 and 128: what the rule for a model lets through, and no kernel beside it."""
    forms = {s[s.index("I") + 1:s.index("EE")] for s in listing if kernel_name(s) == "k_decode_ranks"}
    assert forms == {"fLi64", "tLi64", "tLi128"}


def test_tiles_of_four_stages_exist_for_halves_only(listing):
    """No model multiplies bf16 operands (they become scaled halves at finalize), and planes take two or three stages."""
    forms = {s[s.index("I") + 1:s.index("EE")] for s in listing if kernel_name(s) == "k_gemm_tile"}
    assert {f.split("Li")[0] for f in forms if f.split("Li")[4] == "4E"} == {"5f16_t"}, forms


@pytest.mark.parametrize("hd", [64, 128])
def test_scaled_queries_are_rounded_once(listing, hd):
    """The prefill attention of halves scales its queries in fp32 and rounds to halves: HD / 2 of them a lane, each in one instruction."""
    code = [code for s, code in listing.items() if kernel_name(s) == "k_pf_attn_mfma" and f"Li{hd}E" in s]
    assert len(code) == 2
    for c in code:
        assert sum(bool(re.match(r"v_(fma|mad)_mix(lo|hi)_f16", ins)) for ins in c) >= hd // 2


def test_untagged_operands_are_read_past_the_l1(listing):
    """k_decode_wide reads planes and partial sums that other workgroups of the XCD have stored, behind flags and without tags of their own.  Each of the five
    products that does (first phase, output projection, gate / up, down projection, LM head) drops the compute unit's L1 lines once its flags are there."""
    forms = {s: code for s, code in listing.items() if kernel_name(s) == "k_decode_wide"}
    assert len(forms) == 4
    for symbol, code in forms.items():
        drops = [i for i, ins in enumerate(code) if ins.startswith("buffer_inv sc0") and "sc1" not in ins]
        assert len(drops) >= 5, (symbol, len(drops))
