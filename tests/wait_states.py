"""Wait states between a matrix instruction and the first use of its result, read from a kernel's listing.

The hardware does not hold an instruction back until a matrix instruction's result is in its register: the compiler counts the
instructions between the two and fills up with s_nop. It does not look into inline assembly, so where assembly reads such a result, or
is the matrix instruction, the source has to see to the distance; `early_uses` finds where it does not. Distances are counted as the
compiler counts them: an instruction is one wait state, `s_nop n` is n + 1, whatever a later instruction may itself wait for."""
import re


def registers(operand):
    """Vector registers that an operand names: {("v", n), ..} or {("a", n), ..}."""
    m = re.fullmatch(r"[-|]*([va])(?:\[(\d+):(\d+)\]|(\d+))\|?", operand)
    if not m:
        return set()
    return {(m[1], i) for i in (range(int(m[2]), int(m[3]) + 1) if m[2] else [int(m[4])])}


def wait_states(op, line):
    """What the compiler for gfx950 keeps between this matrix instruction and a vector or memory instruction on its result:
    passes of four cycles and four more."""
    if op in ("v_mfma_f32_16x16x32_bf16",):
        return 8
    if op in ("v_mfma_f32_32x32x16_bf16",):
        return 12
    narrow = "cbsz:4" in line and "blgp:4" in line  # fp4 operands on both sides take half of the passes
    if op == "v_mfma_scale_f32_16x16x128_f8f6f4":
        return 8 if narrow else 12
    if op == "v_mfma_scale_f32_32x32x64_f8f6f4":
        return 12 if narrow else 20
    raise ValueError(f"no wait states known for {op}")


def blocks_of(body):
    """Basic blocks of a kernel's listing in order: [instructions, where it may go on to]; an instruction is (operation, operands,
    its line, whether it is inline assembly)."""
    blocks, names, by_hand = [[[], []]], {}, False
    for line in body.splitlines():
        by_hand = (by_hand or "#ASMSTART" in line) and "#ASMEND" not in line
        text = line.split(";")[0].strip()
        label = re.match(r"(\.?\w+):", text)
        if label:
            blocks.append([[], []])
            names[label[1]] = len(blocks) - 1
            continue
        if not text or text.startswith("."):
            continue
        op, _, rest = text.partition(" ") if "\t" not in text else text.partition("\t")
        args = [a.split()[0] for a in rest.split(",") if a.strip()]
        blocks[-1][0].append((op, args, text, by_hand))
        if op.startswith(("s_branch", "s_cbranch", "s_endpgm")):
            blocks.append([[], []])
    for i, (instructions, to) in enumerate(blocks):
        last = instructions[-1][0] if instructions else ""
        if last.startswith(("s_branch", "s_cbranch")):
            to.append(names[instructions[-1][1][0]])
        if not last.startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            to.append(i + 1)
    return blocks


def early_uses(body):
    """(matrix instructions seen, [(line, wait states missing)]): vector and memory instructions that read a matrix
    instruction's result, or write over it, before its wait states have passed on some way through the kernel."""
    blocks = blocks_of(body)
    entry = [{} for _ in blocks]  # register -> wait states still to pass
    seen, early, again = 0, {}, list(range(len(blocks)))
    while again:
        i = again.pop()
        left = dict(entry[i])
        for op, args, line, _ in blocks[i][0]:
            if op.startswith("v_mfma"):
                passed = 1
            else:
                passed = int(args[0], 0) + 1 if op == "s_nop" else 1
                if op.startswith(("v_", "ds_", "global_", "buffer_", "scratch_", "flat_")):
                    for a in args:
                        short = max((left.get(r, 0) for r in registers(a)), default=0)
                        if short:
                            early[line] = max(short, early.get(line, 0))
            left = {r: n - passed for r, n in left.items() if n > passed}
            if op.startswith("v_mfma"):
                left.update(dict.fromkeys(registers(args[0]), wait_states(op, line)))
        for to in blocks[i][1]:
            more = {r: n for r, n in left.items() if n > entry[to].get(r, 0)}
            if more:
                entry[to].update(more)
                again.append(to)
    seen = sum(op.startswith("v_mfma") for b in blocks for op, *_ in b[0])
    return seen, sorted(early.items())


def kernels(listing):
    """(mangled name, listing) of every kernel."""
    return re.findall(r"^(_Z\w+):(.*?)^\.Lfunc_end", listing, re.S | re.M)
