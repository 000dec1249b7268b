#!/usr/bin/env python3
"""Looks for the loads of a batch in the assembly of csrc/matmul_narrow.hip.

The kernels that take X a part at a time wait for a part by the number of loads that were issued after it, which have to be
all that the source says: eight between each `; ask` and the next `; asked`, in one piece of straight code.  Fails the build
otherwise.  Usage: check_narrow_asks.py file.s"""
import re
import sys

LOADS = 8


def main():
    inside, found, bad = None, 0, []
    for number, line in enumerate(open(sys.argv[1]), 1):
        text = line.strip()
        if text == "; ask":
            if inside is not None:
                bad.append("%d: a batch inside another" % number)
            inside = 0
        elif text == "; asked":
            found += 1
            if inside != LOADS:
                bad.append("%d: %s loads, %d are wanted" % (number, inside, LOADS))
            inside = None
        elif inside is not None:
            if re.match(r"(global|flat|buffer)_load_(dword|ushort)\b", text):
                inside += 1
            elif re.match(r"s_cbranch|s_branch|s_setpc|s_endpgm|[.\w$]+:", text):
                bad.append("%d: a batch's loads are not straight code: %s" % (number, text))
    if inside is not None or found == 0:
        bad.append("no whole batch found")
    for b in bad:
        print("%s:%s" % (sys.argv[1], b), file=sys.stderr)
    return 1 if bad else 0


sys.exit(main())
