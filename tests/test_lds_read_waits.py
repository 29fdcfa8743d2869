"""The MLA prefill kernel reads V out of LDS in assembly, four operands ahead, with the waits written out: to the compiler a
read's registers hold their values at once.  Nothing may touch them before the wait: not a copy, not a spill, not another
variable placed there.  The compiler's output for every instantiation is followed along all its branches for that."""
import os
import re
import shlex
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-metax_amd", "csrc")
TRANSPOSING = "ds_read_b64_tr_b16"


def _device_assembly(name, tmp_path):
    """What the compiler makes of csrc/<name>.hip for the GPU, with the flags the library is built with."""
    lines = subprocess.run(["make", "-n", "-B", f"build/{name}.o"], cwd=CSRC, capture_output=True, text=True, check=True).stdout
    cmd = shlex.split(next(line for line in lines.splitlines() if f"{name}.hip" in line))
    if not os.access(cmd[0], os.X_OK):
        pytest.skip("no hipcc")
    out = tmp_path / f"{name}.s"
    cmd[cmd.index("-o") + 1] = str(out)
    cmd[cmd.index("-c")] = "-S"
    subprocess.run(cmd + ["--cuda-device-only"], cwd=CSRC, capture_output=True, check=True)
    return out.read_text()


def _kernels(text):
    """{name: [(label or None, instruction or None)]} of an assembly file."""
    kernels, body = {}, None
    for line in text.splitlines():
        line = line.split(";")[0].rstrip()
        label = re.fullmatch(r"([.\w$]+):", line)
        if label and label[1].startswith("_Z"):
            body = kernels.setdefault(label[1], [])
        elif label and label[1].startswith(".Lfunc_end"):
            body = None
        elif body is not None and label:
            body.append((label[1], None))
        elif body is not None and re.match(r"\s+[a-z]\w+", line):
            body.append((None, line.strip()))
    return {k: b for k, b in kernels.items() if any(i and i.startswith("ds_read") for _, i in b)}


def _registers(operands):
    regs = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", operands):
        regs.update((kind, r) for r in range(int(lo or one), int(hi or one) + 1))
    return regs


def _early_uses(body):
    """The instructions that touch a register whose LDS read may still be under way.

    Followed per place: {register: LDS operations issued after its read, at least}.  LDS answers in order, so a wait for
    n or fewer outstanding operations ends every read with n or more behind it; scalar loads count for the hardware's
    counter but answer in any order, so they are not counted as being behind a read."""
    at = {label: i for i, (label, _) in enumerate(body) if label}
    before, work, found = {0: {}}, [0], set()
    while work:
        i = work.pop()
        pending = dict(before[i])
        text = body[i][1] or ""
        op, _, operands = text.partition(" ") if " " in text else text.partition("\t")
        if _registers(operands) & pending.keys():
            found.add(i)
            pending = {r: n for r, n in pending.items() if r not in _registers(operands)}
        if op.startswith("ds_"):
            pending = {r: n + 1 for r, n in pending.items()}
            if op.startswith("ds_read"):
                pending.update((r, 0) for r in _registers(operands.split(",")[0]))
        wait = re.search(r"lgkmcnt\((\d+)\)", operands) if op == "s_waitcnt" else None
        if wait:
            pending = {r: n for r, n in pending.items() if n < int(wait[1])}
        after = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if op == "s_branch" or op.startswith("s_cbranch"):
            after.append(at[operands.strip()])
        for j in after:
            if j >= len(body):
                continue
            old = before.get(j)
            new = pending if old is None else {r: min(old.get(r, 1 << 20), pending.get(r, 1 << 20)) for r in old.keys() | pending.keys()}
            if new != old:
                before[j] = new
                work.append(j)
    return [body[i][1] for i in sorted(found)]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    return _kernels(_device_assembly("kvq_mla_prefill", tmp_path_factory.mktemp("asm")))


def test_no_register_of_a_v_read_is_touched_before_its_wait(kernels):
    assert len(kernels) == 6, list(kernels)   # two types, three head shapes
    for name, body in kernels.items():
        assert sum(i is not None and i.startswith(TRANSPOSING) for _, i in body) >= 16, name   # two steps of four blocks or more, two halves
        assert _early_uses(body) == [], name


def test_a_copy_a_reuse_and_a_late_wait_are_seen(kernels):
    """The check finds what it is there for: each of these in one kernel's text."""
    body = next(iter(kernels.values()))
    first = next(i for i, (_, t) in enumerate(body) if t and t.startswith(TRANSPOSING))
    reg = re.search(r"v\[(\d+):", body[first][1])[1]
    waits = [i for i, (_, t) in enumerate(body) if i > first and t and re.fullmatch(r"s_waitcnt lgkmcnt\([1-9]\d*\)", t)]
    for extra in (f"v_mov_b32_e32 v255, v{reg}", f"v_mov_b32_e32 v{reg}, 0", f"scratch_store_dword off, v{reg}, s0"):
        assert extra in _early_uses(body[:first + 1] + [(None, extra)] + body[first + 1:])
    n = int(re.search(r"\((\d+)\)", body[waits[0]][1])[1])
    late = body[:waits[0]] + [(None, f"s_waitcnt lgkmcnt({n + 1})")] + body[waits[0] + 1:]
    assert _early_uses(late) != []
