"""Loads that go straight into LDS (``global_load_lds``) are counted by ``vmcnt``, and a workgroup barrier does not wait
for them: a wave has to, before the barrier that hands what it fetched to the other waves, and before it ends (its LDS is
given back then).  Late data shows only now and then, as wrong values, so this is checked in the code that the library's
own flags make, on every path through every kernel."""
import os
import re
import subprocess

from poker2_amd import build


def assembly(source: str, out: str) -> str:
    flags = [f for f in build.HIPCC_FLAGS if f != "-shared"]
    subprocess.run([build.hipcc_path(), *flags, "--offload-device-only", "-S", "-x", "hip", "-o", out, source], check=True,
                   capture_output=True)
    with open(out) as f:
        return f.read()


def blocks_of(body: list[str]) -> tuple[dict[str, list[str]], dict[str, list[str]]]:
    """Basic blocks of a function's lines, and the blocks that follow each of them."""
    code, nexts, name = {"entry": []}, {"entry": []}, "entry"
    open_block = True                          # whether control can fall out of the block
    for line in body:
        label = re.match(r"(\.LBB\w+):", line)
        if label:
            if open_block:
                nexts[name].append(label[1])
            name, open_block = label[1], True
            code[name], nexts[name] = [], []
            continue
        words = line.split(";")[0].split()
        if not words or words[0].startswith(".") or words[0].endswith(":") or not open_block:
            continue
        code[name].append(" ".join(words))
        if words[0] == "s_branch" or words[0].startswith("s_cbranch"):
            nexts[name].append(words[1])
        if words[0].startswith("s_cbranch"):       # what comes next is another block: it may be skipped
            after = f"{name}|{len(code)}"
            nexts[name].append(after)
            name, code[after], nexts[after] = after, [], []
        assert words[0] not in ("s_setpc_b64", "s_swappc_b64", "s_call_b64"), "a call: not followed here"
        if words[0] in ("s_branch", "s_endpgm"):
            open_block = False
    return code, nexts


def unawaited(body: list[str]) -> list[str]:
    """Barriers and ends of the program that some path reaches with a direct load under way."""
    code, nexts = blocks_of(body)
    reached, todo, found = set(), [("entry", False)], []
    while todo:
        at = todo.pop()
        if at in reached:
            continue
        reached.add(at)
        name, pending = at
        for k, ins in enumerate(code[name]):
            if "load_lds" in ins or ins.endswith(" lds"):
                pending = True
            elif ins.startswith("s_waitcnt") and "vmcnt(0)" in ins:
                pending = False
            elif pending and ins.split()[0] in ("s_barrier", "s_endpgm"):
                found.append(f"{name} + {k}: {ins}")
        todo += [(n, pending) for n in nexts[name]]
    return found


def functions(text: str) -> dict[str, list[str]]:
    out = {}
    for m in re.finditer(r"^(\w+):.*?$(.*?)^\.Lfunc_end", text, re.S | re.M):
        out[m[1]] = m[2].splitlines()
    return out


def test_the_check_itself():
    loop = ["global_load_lds_dwordx4 v1, s[0:1]", ".LBB0_1:", "{wait}", "s_barrier", "global_load_lds_dwordx4 v1, s[0:1]",
            "s_cbranch_execz .LBB0_2", "; %bb.3:", "s_waitcnt vmcnt(0)", "global_store_dword v[0:1], v2, off", ".LBB0_2:",
            "s_cbranch_scc1 .LBB0_1", "; %bb.4:", "{end}", "s_endpgm"]

    def found(wait, end):
        return unawaited([line.format(wait=wait, end=end) for line in loop])
    assert found("s_waitcnt vmcnt(0) lgkmcnt(0)", "s_waitcnt vmcnt(0)") == []
    assert found("s_waitcnt lgkmcnt(0)", "s_waitcnt vmcnt(0)")       # the wait in the loop may be skipped
    assert found("s_waitcnt vmcnt(0)", "s_waitcnt vmcnt(1)")


def test_no_barrier_hands_over_a_load_that_is_still_under_way(tmp_path):
    source = os.path.join(build.CSRC, "leaf_network.hip")
    kernels = {name: body for name, body in functions(assembly(source, str(tmp_path / "leaf_network.s"))).items()
               if any("load_lds" in line for line in body)}
    assert len([k for k in kernels if "ln_gemm" in k]) >= 8 and any("ln_first" in k for k in kernels)
    assert {k: unawaited(body) for k, body in kernels.items()} == {k: [] for k in kernels}


def test_only_the_checked_file_makes_such_loads():
    for name in sorted(os.listdir(build.CSRC)):
        with open(os.path.join(build.CSRC, name)) as f:
            assert name == "leaf_network.hip" or "load_lds" not in f.read(), name
