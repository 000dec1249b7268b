"""check_quad_ring.py matmul_quad.s: the quad-union kernel's register ring, in the compiler's assembly of csrc/matmul_quad.hip.

Loads into v84 .. v95 are in flight while the code between the kernel's inline-assembly blocks runs, and the waits inside
the blocks count the vector memory instructions issued since.  The compiler knows neither, so the build checks what it
made: on every way from the block marked "ring: first requests" to the one marked "ring: drained", no instruction outside
the blocks names one of those registers or is a vector memory instruction.  A copy or a spill in between would read a
value that has not arrived."""
import re
import sys

RING = set(range(84, 96))


def registers(text):
    for lo, hi in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        yield from range(int(lo), int(hi) + 1)
    for r in re.findall(r"\bv(\d+)\b", text):
        yield int(r)


def kernels(lines):
    """(name, its lines) of every quad-union kernel."""
    name = None
    for line in lines:
        start = re.match(r"(\S*ellpack_matmul_quad_kernel\S*):", line)
        if start:
            name, body = start.group(1), []
        elif name and line.startswith(".Lfunc_end"):
            yield name, body
            name = None
        elif name:
            body.append(line)


def instructions(body):
    """[('asm', text) | ('op', text)], {label: index}; an inline-assembly block is one instruction."""
    out, labels, block = [], {}, None
    for line in body:
        if ";#ASMSTART" in line:
            block = []
        elif ";#ASMEND" in line:
            out.append(("asm", "\n".join(block)))
            block = None
        elif block is not None:
            block.append(line)
        else:
            text = line.split(";")[0].strip()
            label = re.match(r"(\.L\w+):", text)
            if label:
                labels[label.group(1)] = len(out)
            elif text and not text.startswith("."):
                out.append(("op", text))
    return out, labels


def check(body):
    code, labels = instructions(body)
    first = [i for i, (k, t) in enumerate(code) if k == "asm" and "ring: first requests" in t]
    last = {i for i, (k, t) in enumerate(code) if k == "asm" and "ring: drained" in t}
    if len(first) != 1 or not last:
        return ["the marked blocks are missing"]
    faults, seen, todo = [], set(), [first[0] + 1]
    while todo:
        i = todo.pop()
        if i in seen or i in last:
            continue
        seen.add(i)
        kind, text = code[i]
        if kind == "op":
            op, _, args = text.partition(" ")
            if op in ("s_endpgm", "s_setpc_b64", "s_swappc_b64"):
                faults.append("leaves the kernel's body with the ring in flight: " + text)
                continue
            if op == "s_branch":
                todo.append(labels[args.strip()])
                continue
            if op.startswith("s_cbranch"):
                todo.append(labels[args.strip()])
            if RING.intersection(registers(text)):
                faults.append("names a ring register: " + text)
            if re.match(r"(global|buffer|flat|scratch|image)_", op):
                faults.append("a vector memory instruction between the blocks: " + text)
        todo.append(i + 1)
    return faults


def main(path):
    found = 0
    for name, body in kernels(open(path).read().splitlines()):
        found += 1
        faults = check(body)
        if faults:
            sys.exit("%s: %s" % (name, "; ".join(faults)))
    if not found:
        sys.exit("no quad-union kernel in " + path)


if __name__ == "__main__":
    main(sys.argv[1])
