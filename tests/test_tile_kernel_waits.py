"""The prompt tile kernel's counted waits against the loads that the compiler emitted.

gemm_tile.h waits for a stage of token rows by counting the vector loads behind it: the next stage's and at least one load per row block and part of
weights.  A format whose part load came out as a scalar load, or merged over both row blocks, would leave fewer behind and the barrier would let
waves read rows that have not landed.  Here the gfx950 code of the built library is listed and every wait is checked against its loop."""
import re
import subprocess
from pathlib import Path

import pytest

from pocketllm_amd import _ffi

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
MOE_FETCH = {"global_load_dwordx4", "global_load_dwordx2", "global_load_ushort"}         # weights: no other load of the routed tiles' loop has these
FORMATS = {"TQ4K", "TQ5K", "TQ2K", "TQ6K", "TIQ4XS", "TIQ2XXS", "TIQ2XS", "TIQ3XXS", "TIQ1M", "TFP8"}
VECTOR_MEMORY = re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)\w*")


def _kernels(tmp_path, marker=b"gemm_tile_kernel", pattern=r"gemm_tile_kernelINS_\d+(\w+?)ELi(\d+)E", key=lambda m: (m[1], int(m[2]))):
    """(format, NT) -> [(address, mnemonic, operands)] of every gemm_tile_kernel (or what `pattern` names) in the library."""
    lib = tmp_path / "lib.so"
    lib.symlink_to(_ffi.LIB_PATH)
    subprocess.run([str(OBJDUMP), "--offloading", str(lib)], check=True, cwd=tmp_path, stdout=subprocess.DEVNULL)
    kernels = {}
    for obj in sorted(tmp_path.glob("lib.so.*gfx950")):
        if marker not in obj.read_bytes():
            continue
        listing = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
        current = None
        for line in listing.splitlines():
            if line.endswith(">:"):
                name = re.search(pattern, line)
                current = kernels.setdefault(key(name), []) if name else None
            elif current is not None and "//" in line:
                text, at = line.split("//", 1)
                mnemonic, _, operands = text.strip().partition(" ")
                target = re.search(r"\+0x([0-9a-f]+)>", at)
                current.append((int(at.split(":")[0], 16), mnemonic, operands, int(target[1], 16) if target else None))
    return kernels


def _vmcnt(operands):
    found = re.search(r"vmcnt\((\d+)\)", operands)
    return int(found[1]) if found else None


def _faults(code, nt):
    """What is wrong with the waits of one kernel, as texts."""
    start, index = code[0][0], {at: i for i, (at, *_) in enumerate(code)}
    loops = []
    for i, (at, mnemonic, _, offset) in enumerate(code):
        if mnemonic.startswith(("s_cbranch", "s_branch")) and offset is not None and start + offset < at and start + offset in index:
            body = code[index[start + offset]:i]
            if sum(m == "s_barrier" for _, m, *_ in body) == 4:
                loops.append((index[start + offset], body))
    if not loops:
        return ["no loop of four steps"]
    first, body = min(loops, key=lambda l: len(l[1]))

    def events(part):                              # "T": a token load, "W": any other vector memory instruction, a count: a wait, "B": a barrier
        out = []
        for _, m, operands, _ in part:
            if m == "global_load_lds_dwordx4":
                out.append("T")
            elif VECTOR_MEMORY.fullmatch(m):
                out.append("W" if "_load" in m and not m.startswith("scratch") else "?")
            elif m == "s_waitcnt" and _vmcnt(operands) is not None:
                out.append(_vmcnt(operands))
            elif m == "s_barrier":
                out.append("B")
        return out

    faults, round_ = [], events(body)
    if "?" in round_:
        faults.append("stores, atomics or spills in the loop")
    if round_.count("T") != 4 * nt:
        faults.append(f"{round_.count('T')} token loads in four steps")
    twice = round_ + round_
    for at, event in enumerate(twice):
        if event != "B" or at < len(round_):
            continue
        # the stage that is read behind this barrier: the last but one whose loads stand before it; waits between them may each cover it
        tokens, covered, behind, seen = 0, False, 0, []
        for e in reversed(twice[:at]):
            if e == "T":
                tokens += 1
                if tokens > nt:
                    break
                behind += 1
            elif e in ("W", "?"):
                behind += 1
            elif isinstance(e, int):
                seen.append((e, behind))
        covered = any(count <= behind - later for count, later in seen)
        if not covered:
            faults.append(f"a step's rows have {behind} loads behind them, waits {seen}")
    # before the loop: all three stages have landed at the last barrier
    ahead = events(code[:first])
    ahead = ahead[:len(ahead) - ahead[::-1].index("B")]
    last = len(ahead) - 1 - ahead[::-1].index("T")
    behind, landed = 0, False
    for e in ahead[last + 1:]:
        behind += e == "W"
        landed |= isinstance(e, int) and e <= behind
    if not landed:
        faults.append("the first stages are not waited for")
    return faults


@pytest.mark.skipif(not _ffi.LIB_PATH.exists() or not OBJDUMP.exists(), reason="needs the built library and ROCm's llvm-objdump")
def test_counted_waits_of_the_tile_kernel(tmp_path):
    kernels = _kernels(tmp_path)
    assert set(kernels) == {(f, nt) for f in FORMATS for nt in (1, 2, 4, 8)} - {("TFP8", 1)}
    wrong = {key: faults for key, code in kernels.items() if (faults := _faults(code, key[1]))}
    assert not wrong
    # the check itself: with one part's loads made scalar, or the loads of both row blocks one, the same loop fails
    code = kernels["TQ4K", 4]
    weights = [i for i, (_, m, *_) in enumerate(code) if m == "global_load_dwordx4"]
    for keep in (0, 1):
        fewer = [(a, "s_nop" if i in weights and weights.index(i) % 2 >= keep else m, o, t) for i, (a, m, o, t) in enumerate(code)]
        assert _faults(fewer, 4)


def _moe_gates(code):
    """Of every counted wait in front of a barrier in the routed experts' tile kernel: (count, weight loads behind the last direct-to-LDS load)."""
    start, index = code[0][0], {at: i for i, (at, *_) in enumerate(code)}
    loops = [(index[start + offset], i) for i, (at, m, _, offset) in enumerate(code)
             if m.startswith(("s_cbranch", "s_branch")) and offset is not None and start + offset < at and start + offset in index]
    gates = []
    for i, (_, m, operands, _) in enumerate(code):
        count = _vmcnt(operands) if m == "s_waitcnt" else None
        if not count or all(later != "s_barrier" for _, later, *_ in code[i + 1:i + 4]):
            continue
        first, last = min((l for l in loops if l[0] <= i <= l[1]), key=lambda l: l[1] - l[0])      # the loop over the blocks
        behind = 0
        for _, earlier, *_ in reversed(code[i:last + 1] + code[first:i]):                          # (once around)
            if earlier == "global_load_lds_dwordx4":
                break
            behind += earlier in MOE_FETCH
        else:
            behind = None
        gates.append((count, behind))
    return gates


@pytest.mark.skipif(not _ffi.LIB_PATH.exists() or not OBJDUMP.exists(), reason="needs the built library and ROCm's llvm-objdump")
def test_counted_waits_of_the_routed_tiles(tmp_path):
    """Tiles of up to 64 rows wait at every other gate for the activations but not for the weights that were asked for behind them."""
    kernels = _kernels(tmp_path, b"moe_tile_kernel", r"moe_tile_kernelINS\d*_\d+Tile(\w+?)ELb(\d)ELi(\d)ELb", lambda m: (m[1], int(m[2]), int(m[3])))
    assert set(kernels) == {(f, small, t) for f, terms in (("IQ2XXS", (1, 2)), ("IQ1M", (1,))) for t in terms for small in (0, 1)}
    for (fmt, small, _), code in kernels.items():
        gates = _moe_gates(code)
        assert len(gates) == (0 if small else 2), (fmt, small, gates)                              # (one per height of the tile)
        assert all(behind is not None and count <= behind for count, behind in gates), (fmt, gates)
    fewer = [(a, "s_nop" if m == "global_load_ushort" else m, o, t) for a, m, o, t in kernels["IQ2XXS", 0, 1]]
    assert any(count > behind for count, behind in _moe_gates(fewer))


# weight loads of a step of the rows kernel: pieces (16 bytes), and the tail's forms (one is executed: blocks that start between two words or on one)
ROWS = {"Q6K": (7, {"global_load_ushort", "global_load_dword"}), "IQ4XS": (4, {"global_load_dwordx2"}), "Q2K": (3, {"global_load_dword"})}


def _rows_faults(code, pieces, tails):
    """What is wrong with the waits in front of the rows kernel's barriers: the step's activations have as many loads behind them as the wait leaves."""
    faults, gates = [], 0
    for i, (_, m, *_) in enumerate(code):
        if m != "s_barrier":
            continue
        gates += 1
        step = code[:i]
        step = step[len(step) - [e[1] for e in reversed(step)].index("global_load_lds_dwordx4"):]      # from the last activation load to the barrier
        behind, landed = [], False
        for _, earlier, operands, _ in step:
            behind.append(earlier)
            if earlier == "s_waitcnt" and (count := _vmcnt(operands)) is not None:
                landed |= count <= behind.count("global_load_dwordx4") + all(t in behind for t in tails)
        if behind.count("global_load_dwordx4") % pieces or not behind.count("global_load_dwordx4"):
            faults.append(f"{behind.count('global_load_dwordx4')} loads of pieces")
        if not all(t in behind for t in tails):
            faults.append(f"tails by {sorted(tails & set(behind))}")
        if not landed:
            faults.append(f"no wait for the activations ahead of {behind.count('global_load_dwordx4')} pieces and {sorted(tails & set(behind))}")
        if any(e.startswith(("scratch", "buffer", "flat")) or "store" in e for e in behind):
            faults.append("stores or spills in the loop")
    return faults if gates == 3 else [*faults, f"{gates} gates"]                     # ahead of the loop, and of its two steps


@pytest.mark.skipif(not _ffi.LIB_PATH.exists() or not OBJDUMP.exists(), reason="needs the built library and ROCm's llvm-objdump")
def test_counted_waits_of_the_rows_kernel(tmp_path):
    """Between decode and prompts a step waits for its activation rows but not for the weights of two steps ahead that were asked for behind them, on either
    side of the branch of Q6_K's tails."""
    kernels = _kernels(tmp_path, b"kquant_rows_kernel", r"kquant_rows_kernelINS\d*_\d+Rows(\w+?)ELi(\d)ELi(\d)ELi(\d+)E", lambda m: (m[1], *map(int, m.groups()[1:])))
    assert set(kernels) == {("Q6K", 1, 1, 8), *(("Q6K", mb, t, s) for mb, s in ((1, 16), (1, 32), (2, 0)) for t in (1, 2)),
                            *(("IQ4XS", mb, t, s) for mb, s in ((1, 16), (1, 32), (2, 64)) for t in (1, 2)), *(("Q2K", mb, t, 0) for mb in (1, 2) for t in (1, 2))}
    wrong = {key: faults for key, code in kernels.items() if (faults := _rows_faults(code, *ROWS[key[0]]))}
    assert not wrong
    # the check itself: without one form of the tail, or without a piece
    for key, lost in ((("Q6K", 1, 1, 8), "global_load_ushort"), (("Q6K", 1, 1, 16), "global_load_dword"), (("IQ4XS", 2, 1, 64), "global_load_dwordx2")):
        assert _rows_faults([(a, "s_nop" if m == lost else m, o, t) for a, m, o, t in kernels[key]], *ROWS[key[0]])
    one = next(i for i, (_, m, *_) in enumerate(kernels["Q2K", 1, 1, 0]) if m == "global_load_dwordx4")
    assert _rows_faults([(a, "s_nop" if i == one else m, o, t) for i, (a, m, o, t) in enumerate(kernels["Q2K", 1, 1, 0])], *ROWS["Q2K"])
