"""The fused GEMMs stage their activation / dY tile by LDS DMA written as inline assembly, which
the compiler does not count, and wait for it with an explicit `s_waitcnt vmcnt(N)`: that is
right only if at least N other vector-memory loads are issued after a step's DMA and before the
wait (loads complete in order, so vmcnt(N) leaves only the N youngest in flight).  This test
compiles nf4_gemm.hip for gfx950 to assembly (hipcc cross-compiles without a GPU) and checks,
in every forward and input-gradient kernel, that after each group of `buffer_load_dwordx4 ...
lds` instructions a wait that covers it comes before the next barrier.

The dense kernel of nf4_dense.hip waits by hand-counted groups whose loads stay in flight over
several barriers, with two wave groups one segment apart.  For it the instruction stream is
checked to be the counted one (only DMA between the prologue and the last wait, nothing spilled
to memory), and the schedule itself is replayed in a model of both wave groups: everything read
has arrived in every wave a barrier before, and nothing is overwritten that may still be read.

A load written as inline assembly is not known to the compiler at all: it neither waits for it
nor knows that its destination registers are busy until the explicit wait.  A second test
replays every kernel's instruction stream (each loop body twice, the second pass starting with
the loads still in flight at the end of the first; a forward branch hands its state to its
target) through an in-order model of the vmcnt counter and checks that no instruction reads or
writes a register that an inline-assembly load still in flight is to write."""

import re

import pytest



def _kernels(asm: str):
    """(name, lines) of every function in the assembly text; an instruction written as inline
    assembly in the source (between the compiler's ASMSTART / ASMEND markers) gets the prefix
    "@asm ".  """
    out, name, body, in_asm = [], None, [], False
    for line in asm.split("\n"):
        m = re.match(r"^(_Z\S+):", line)
        if m:
            name, body = m.group(1), []
            continue
        if name is None:
            continue
        if line.startswith(".Lfunc_end"):
            out.append((name, body))
            name = None
            continue
        if ";;#ASMSTART" in line:
            in_asm = True
        elif ";;#ASMEND" in line:
            in_asm = False
        t = line.split(";")[0].strip()
        if t:
            body.append(("@asm " + t) if in_asm else t)
    return out


def _strip(lines):
    return [t[5:] if t.startswith("@asm ") else t for t in lines]


def _is_dma(t):
    return t.startswith("buffer_load_dwordx4") and t.endswith(" lds")


def _check(lines, barriers_allowed=0):
    """Number of DMA groups checked; raises AssertionError on a group not covered by a wait
    before barrier number barriers_allowed + 1 after it."""
    groups, i, n = 0, 0, len(lines)
    while i < n:
        if not _is_dma(lines[i]):
            i += 1
            continue
        # the group: DMA instructions with no other load, wait, barrier or branch between them
        j, k = i, i + 1
        while k < n and (_is_dma(lines[k]) or not (
                lines[k].startswith(("buffer_load", "global_load", "s_barrier", "s_cbranch",
                                     "s_branch", "s_endpgm", "."))
                or lines[k].startswith("s_waitcnt") and "vmcnt" in lines[k])):
            if _is_dma(lines[k]):
                j = k
            k += 1
        groups += 1
        loads, covered, barriers = 0, False, 0
        for t in lines[j + 1:]:
            if t.startswith(("buffer_load", "global_load")):
                loads += 1
            elif t.startswith("s_waitcnt") and "vmcnt(" in t:
                if int(re.search(r"vmcnt\((\d+)\)", t).group(1)) <= loads:
                    covered = True
                    break
            elif t.startswith("s_barrier"):
                barriers += 1
                if barriers > barriers_allowed:
                    break
        assert covered, f"DMA group ending at line {j} is not waited for in time"
        i = j + 1
    return groups


@pytest.fixture(scope="module")
def kernels(gemm_asm):
    """(name, lines) of every forward and input-gradient kernel of nf4_gemm.hip."""
    ks = [(k, b) for k, b in _kernels(gemm_asm) if re.search(r"(fwd|dx)_(head_tail_|rw_)?kernel", k)]
    assert len(ks) >= 8
    return ks


_REG = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        if m.group(3) is not None:
            out.add(int(m.group(3)))
        else:
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def _replay(lines):
    """In-order vmcnt model over the instruction stream.  Loads written as inline assembly
    ("@asm " lines) are tracked with their destination registers (the compiler waits for its own
    loads before their registers are touched); every load and store counts in vmcnt.  Control
    flow: a forward branch hands its states (the possible queues of loads in flight) to its
    target label, an unconditional one ends the fall-through path, and a backward branch (a loop)
    replays the loop body once with the states its first pass ends in.  Returns the hazards
    (line, instruction, register): an instruction that reads or writes a register an assembly
    load still in flight is to write."""
    labels = {t[:-1]: i for i, t in enumerate(lines) if t.startswith(".L") and t.endswith(":")}
    hazards = []

    def flag(i, t, regs, queues):
        for r in regs:
            if any(r in q for qu in queues for q in qu):
                hazards.append((i, t, r))

    def step(i, queues):
        """Apply line i to every possible queue; returns the new list of queues."""
        t = lines[i]
        is_asm = t.startswith("@asm ")
        if is_asm:
            t = t[5:]
        op = t.split()[0] if t else ""
        if op.startswith("s_waitcnt") and "vmcnt(" in t:
            keep = int(re.search(r"vmcnt\((\d+)\)", t).group(1))
            return [qu[max(0, len(qu) - keep):] for qu in queues]
        if op.startswith(("buffer_load", "global_load", "buffer_store", "global_store",
                          "buffer_atomic", "global_atomic")):
            ops = t[len(op):]
            dst = frozenset()
            src_txt = ops
            if op.startswith(("buffer_load", "global_load")) and not t.endswith(" lds"):
                dst_txt, src_txt = ops.split(",", 1)
                flag(i, t, _regs(dst_txt), queues)
                if is_asm:
                    dst = frozenset(_regs(dst_txt))
            flag(i, t, _regs(src_txt), queues)
            return [qu + (dst,) for qu in queues]
        flag(i, t, _regs(t), queues)
        return queues

    def dedup(queues):
        return list(dict.fromkeys(queues))

    pending = {}
    states = [()]
    looped = set()
    for i, t in enumerate(lines):
        if t.startswith(".L") and t.endswith(":"):
            states = dedup(states + pending.pop(t[:-1], []))
            continue
        if not states:
            continue
        states = step(i, states)
        if t.startswith(("s_cbranch", "s_branch")):
            target = t.split()[-1]
            start = labels.get(target)
            if start is not None and start > i:
                pending[target] = dedup(pending.get(target, []) + states)
            elif start is not None and target not in looped:
                looped.add(target)
                for k in range(start + 1, i + 1):
                    if not (lines[k].startswith(".L") and lines[k].endswith(":")):
                        states = step(k, states)
                states = dedup(states)
            if t.startswith("s_branch"):
                states = []
        elif t.startswith("s_endpgm"):
            states = []
    return hazards


@pytest.mark.timeout(600)
def test_dma_is_waited_for_before_the_barrier(kernels):
    checked = 0
    for name, body in kernels:
        g = _check(_strip(body))
        assert g >= 3, f"{name}: expected the prologue's and the loop's DMA groups, found {g}"
        checked += g
    assert checked > 0


@pytest.mark.timeout(600)
def test_no_register_of_a_load_in_flight_is_touched(kernels):
    for name, body in kernels:
        hz = _replay(body)
        assert not hz, f"{name}: {hz[:3]}"


@pytest.mark.timeout(600)
def test_m0_is_settled_before_the_dma_reads_it(gemm_asm, dense_asm):
    """LDS DMA takes its LDS address from M0 and needs one wait state after a scalar write of it;
    the compiler puts one after its own writes, an inline-assembly statement has to itself."""
    checked = 0
    for name, body in _kernels(gemm_asm) + _kernels(dense_asm):
        lines = [t for t in _strip(body) if not t.endswith(":")]
        for before, t in zip(lines, lines[1:]):
            if _is_dma(t):
                assert not re.match(r"s_\w+ m0\b", before), f"{name}: {before} / {t}"
                checked += 1
    assert checked > 200


def _dense_tokens(body):
    """[(label or None, [tokens], next labels)] of a kernel's basic blocks, tokens: D (DMA), V
    (other vector memory), w<n> / W<n> (vmcnt(n) without / with lgkmcnt(0)), B, m."""
    blocks, label, toks, out = [], None, [], []
    for t in _strip(body):
        if t.endswith(":"):
            blocks.append((label, toks))
            label, toks = t[:-1], []
        elif _is_dma(t):
            toks.append("D")
        elif re.match(r"(buffer|global|flat|scratch)_", t):
            toks.append("V")
        elif t.startswith("s_waitcnt") and "vmcnt(" in t:
            n = re.search(r"vmcnt\((\d+)\)", t).group(1)
            toks.append(("W" if "lgkmcnt(0)" in t else "w") + n)
        elif t.startswith("s_barrier"):
            toks.append("B")
        elif "_mfma_" in t:
            toks.append("m")
        elif t.startswith(("s_cbranch", "s_branch")):
            toks.append(("jump" if t.startswith("s_branch") else "maybe") + " " + t.split()[-1])
        elif t.startswith("s_endpgm"):
            toks.append("end")
    return blocks + [(label, toks)]


@pytest.mark.timeout(600)
def test_dense_kernel_issues_what_its_waits_count(dense_asm):
    from tests.test_skinny_occupancy import _metadata

    meta = dense_asm[dense_asm.index("amdhsa.kernels:"):]
    names = [n for n in _metadata(dense_asm) if "dense_kernel" in n]
    assert len(names) == 2
    for name in names:
        block = next(b for b in re.split(r"\n  - ", meta) if re.search(rf"\.name:\s+{name}\b", b))
        for key in ("private_segment_fixed_size", "sgpr_spill_count", "vgpr_spill_count"):
            assert re.search(rf"\.{key}:\s+(\d+)", block).group(1) == "0", (name, key)
        blocks = _dense_tokens(dict(_kernels(dense_asm))[name])
        # the counted runs: a tile's prologue and one step, of 256x256 and of 128x128 tiles
        grammar = re.compile(r"(D{12}w6B|D{12}w8B|(D{4}W8Bm{16}BD{4}W6Bm{16}B)+|(D{4}W8Bm{8}B)+)$")
        runs = 0
        for _, toks in blocks:
            if "D" not in toks:
                continue
            run = [t for t in toks if not t.startswith(("jump", "maybe"))]
            if run[:12] == ["D"] * 12:  # (waves 4-7 cross one more barrier in a block of their own)
                run = run[:14]
            assert grammar.match("".join(run)), (name, toks)
            runs += 1
        assert runs >= 6, (name, runs)
        # from a prologue on, no vector memory but DMA before vmcnt(0), on any way through
        at = {label: i for i, (label, _) in enumerate(blocks)}
        todo = [i for i, (_, toks) in enumerate(blocks) if toks[:12] == ["D"] * 12]
        seen = set()
        while todo:
            i = todo.pop()
            if i in seen:
                continue
            seen.add(i)
            through = True
            for t in blocks[i][1]:
                assert t not in ("V", "end"), (name, blocks[i])
                if t in ("w0", "W0"):
                    through = False
                    break
                if t.startswith(("jump", "maybe")):
                    todo.append(at[t.split()[1]])
                    if t.startswith("jump"):
                        through = False
                        break
            if through:
                todo.append(i + 1)


# The schedule of dense_tile (nf4_dense.hip) as one wave group runs it: ("send", half, step),
# ("read", half, step), ("wait", n) for vmcnt(n) lgkmcnt(0), "barrier".  Halves: w0, w1 (rows p),
# x0, x1 (rows m); a send is two loads.
def _dense_schedule(big, steps, group):
    if big:
        prologue = [("w0", 0), ("x0", 0), ("x1", 0), ("w1", 0), ("w0", 1), ("x0", 1)]
        first = 6
    else:
        prologue = [(h, u) for u in range(3) for h in ("w0", "x0")]
        first = 8
    ops = [("send", h, u) for h, u in prologue] + [("wait", first), "barrier"]
    ops += ["barrier"] * group
    for u in range(steps):
        if big:
            ops += [("read", h, u) for h in ("x0", "x1", "w0")]
            ops += [("send", "x1", u + 1), ("send", "w1", u + 1), ("wait", 8), "barrier", "barrier",
                    ("read", "w1", u), ("send", "w0", u + 2), ("send", "x0", u + 2), ("wait", 6),
                    "barrier", "barrier"]
        else:
            ops += [("read", "x0", u), ("read", "w0", u), ("send", "w0", u + 3),
                    ("send", "x0", u + 3), ("wait", 8), "barrier", "barrier"]
    return ops + ["barrier"] * (1 - group) + [("wait", 0), "barrier"]


def _dense_hazards(big, steps, schedule=_dense_schedule):
    """Violations in the schedule of both wave groups, barrier to barrier (what two groups do
    between the same barriers is unordered)."""
    stages = 2 if big else 4
    writes, reads, spans = [], [], []
    for group in (0, 1):
        flight, span = [], 0
        for op in schedule(big, steps, group):
            if op == "barrier":
                span += 1
            elif op[0] == "send":
                w = [op[1], op[2] % stages, op[2], span, None]  # half, stage, step, issued, arrived
                writes.append(w)
                flight += [w, w]
            elif op[0] == "read":
                reads.append((op[1], op[2] % stages, op[2], span))
            else:
                done = flight[:max(0, len(flight) - op[1])]
                flight = flight[len(done):]
                for w in done:
                    if w not in flight and w[4] is None:
                        w[4] = span
        spans.append(span)
        assert not flight
    bad = [] if spans[0] == spans[1] else [("barriers", spans)]
    for half, stage, step, span in reads:
        for w in writes:
            if w[:2] != [half, stage]:
                continue
            if w[2] == step and not w[4] < span:
                bad.append(("read before it arrived", half, step, span, w))
            if w[2] > step and not w[3] > span:
                bad.append(("overwritten while it may be read", half, step, span, w))
        assert sum(w[:3] == [half, stage, step] for w in writes) == 2  # both groups' shares
    return bad


@pytest.mark.parametrize("big", [True, False])
def test_dense_schedule_reads_what_arrived(big):
    for steps in range(1, 14):
        assert not _dense_hazards(big, steps), steps


def test_dense_schedule_model_flags_a_missing_wait_and_an_early_send():
    def later_wait(big, steps, group):
        return [("wait", 10) if op == ("wait", 6) else op
                for op in _dense_schedule(big, steps, group)]

    def early_send(big, steps, group):  # x0 two steps ahead while this step's is being read
        swap = {"x1": ("x0", 1), "x0": ("x1", -1)}
        ops, first = _dense_schedule(big, steps, group), 6
        return ops[:first] + [("send", swap[op[1]][0], op[2] + swap[op[1]][1])
                              if op[0] == "send" and op[1] in swap else op for op in ops[first:]]

    assert any("arrived" in b[0] for b in _dense_hazards(True, 5, later_wait))
    assert any("overwritten" in b[0] for b in _dense_hazards(True, 5, early_send))


def test_replay_model_flags_a_register_used_before_its_wait():
    """The model itself: a load whose register is read before a wait covers it is flagged; the
    same read after vmcnt(0), or after a vmcnt(1) that leaves only a younger load in flight, is
    not."""
    base = ["@asm buffer_load_dwordx4 v[4:7], v1, s[0:3], 0 offen",
            "@asm buffer_load_dword v9, v2, s[0:3], 0 offen"]
    assert _replay(base + ["v_add_u32_e32 v10, v5, v3"])
    assert not _replay(base + ["s_waitcnt vmcnt(1)", "v_add_u32_e32 v10, v5, v3"])
    assert _replay(base + ["s_waitcnt vmcnt(1)", "v_add_u32_e32 v10, v9, v3"])
    assert not _replay(base + ["s_waitcnt vmcnt(0)", "v_add_u32_e32 v10, v9, v3"])
    # a loop body replayed: the load issued at its end is in flight at its start
    loop = [".LBB0_1:", "v_mov_b32_e32 v20, v8", "s_waitcnt vmcnt(0)",
            "@asm buffer_load_dword v8, v2, s[0:3], 0 offen", "s_cbranch_scc1 .LBB0_1"]
    assert _replay(loop)
    # the DMA form writes no register (its first operand is the address)
    assert not _replay(["@asm buffer_load_dwordx4 v3, s[0:3], s4 offen lds", "v_mov_b32_e32 v5, v3"])
    # a load the compiler issued is not tracked (the compiler waits for it itself)
    assert not _replay(["buffer_load_dword v9, v2, s[0:3], 0 offen", "v_mov_b32_e32 v5, v9"])
