"""The folded GEMM's waits for its global-to-LDS copies count the vector-memory loads that its code issues
after them; the counts are kept by hand (loads of a unit, of a min-pass record, of a stage's codes).
This follows the built gfx950 code of every mmqh_kernel's loop: at each stage's barrier the wave has
waited for the copies of the next stage, whatever loads the compiler emitted between."""
import re
import shutil
import subprocess

import pytest

import _oracle as O
from test_build_m0 import LIB, OBJDUMP

MIN_SLOTS = {O.Q4_K: 3, O.Q2_K: 4}


def stages_in_lds(qtype, ct, gn, gk, st):
    """NS of MmqhTile."""
    qk, size = O.BLOCK[qtype]
    bm = 32 * ct
    seg = (4 if st == 2 else 4 if qk == 256 else 2) * 64 * size // qk
    raw = gn * 32 * ((seg + 15) // 32 * 32 + 16) if st else 0
    fits = gk * (4 * 128 * bm + 16 * bm * MIN_SLOTS.get(qtype, 0) + raw) <= 160 * 1024
    return 4 if st != 1 and fits else 3


def kernels(tmp_path):
    lib = tmp_path / LIB.name
    shutil.copy(LIB, lib)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    for obj in sorted(tmp_path.glob(f"{LIB.name}.*gfx950")):
        text = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True,
                              text=True).stdout
        name, code = None, []
        for line in text.split("\n") + ["0 <>:"]:
            m = re.match(r"^([0-9a-f]+) <(.*)>:", line)
            if m or line == "0 <>:":
                if name and "mmqh_kernel" in name:
                    yield name, code
                name, code = (m.group(2), []) if m else (None, [])
                continue
            m = re.match(r"^\s+(\S+)\s*(.*?)\s*//\s*([0-9A-F]+):", line)
            if m:
                target = re.search(r"<[^>]*\+0x([0-9a-f]+)>", line)
                code.append((int(m.group(3), 16), m.group(1), m.group(2), target and int(target.group(1), 16)))


def loop_events(code, count):
    """The main loop's `count` copies (C), its other vector-memory accesses (L), vmcnt waits (n) and barriers
    (B) in order."""
    base, at = code[0][0], {c[0]: i for i, c in enumerate(code)}
    copies = [i for i, c in enumerate(code) if c[1] == "global_load_lds_dwordx4"]
    loops = [(at[base + c[3]], i) for i, c in enumerate(code)
             if c[1].startswith(("s_cbranch", "s_branch")) and c[3] is not None and base + c[3] in at and at[base + c[3]] <= i]
    start, end = min((l for l in loops if sum(l[0] <= i <= l[1] for i in copies) == count), key=lambda l: l[1] - l[0])

    def has(a, b, *names):
        return any(c[1] in names for c in code[a:b])

    events, i, steps = [], start, 0
    while i <= end and steps < 20000:
        steps += 1
        _, op, args, target = code[i]
        if op == "global_load_lds_dwordx4":
            events.append("C")
        elif op.startswith(("global_load", "buffer_load", "flat_load", "scratch_load", "global_store", "scratch_store")):
            events.append("L")
        elif op == "s_barrier":
            events.append("B")
        elif op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", args)
            if m:
                events.append(int(m.group(1)))
        if op.startswith(("s_cbranch", "s_branch")) and target is not None:
            j = at[base + target]
            if j > i and (op == "s_branch" or has(i + 1, min(j, end), "s_barrier") and not has(
                    i + 1, min(j, end), "global_load_lds_dwordx4")):
                i = j
                continue
        i += 1
    return events


@pytest.mark.skipif(not LIB.exists() or not OBJDUMP.exists(), reason="needs the built library and llvm-objdump")
def test_waits_cover_the_next_stage(tmp_path):
    seen = 0
    for name, code in kernels(tmp_path):
        qtype, ct, gn, gk, st = (int(v) for v in re.search(r"mmqh_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E",
                                                           name).groups())
        ns = stages_in_lds(qtype, ct, gn, gk, st)
        code_ops = 128 * 32 * ct // (16 * 64 * gn)  # 16-byte copies of a thread and stage
        events = loop_events(code, 4 * code_ops)
        assert events.count("B") == 4 and events.count("C") == 4 * code_ops, (name, events)
        first = events.index("C")
        events = events[first:] + events[:first]  # the loop may be laid out from its middle
        queue, interval, per = [], 0, []  # loads in flight, each with the barrier interval that issued it
        for e in events * 6:
            if e == "C" or e == "L":
                queue.append((e, interval))
                per.append(e)
            elif e == "B":
                assert per.count("C") == code_ops, (name, interval)
                # barrier s: the copies of stage s + 1 were issued in interval s + 2 - ns
                late = [q for q in queue if q[0] == "C" and q[1] <= interval + 2 - ns]
                assert not late, (name, interval, late)
                interval, per = interval + 1, []
            else:
                queue = queue[len(queue) - e:] if len(queue) > e else queue
        seen += 1
    assert seen == 50
