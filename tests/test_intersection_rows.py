"""A team's rows of path terms: the first term's high word tells a longer piece's
row (its vertices and ends follow) from terms.  A vertex may hold any NaN, whose
low bits the widening to 64 bits and the products keep, so a NaN term is stored
as the one quiet NaN.  The kernel's steps are restated in C here, with the mark
read from its source."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
static uint32_t high(double v) { uint64_t b; memcpy(&b, &v, 8); return (uint32_t)(b >> 32); }
int main(int argc, char **argv) {
    const uint32_t mark = (uint32_t)strtoul(argv[1], NULL, 16);
    long plain = 0, stored = 0;
    for (uint32_t low = 0; low < 1u << 23; low++)
        for (uint32_t sign = 0; sign < 2; sign++) {
            const uint32_t b = sign << 31 | 0x7f800000u | low;  /* every NaN, and infinity */
            volatile float x;
            memcpy((void *)&x, &b, 4);
            double t = ((double)x - 0.25) * (1.5 - 0.5) - (2.5 - 0.25) * (3.5 - 0.5);
            plain += high(t) == mark;
            GUARD
            stored += high(t) == mark;
        }
    printf("%ld %ld\n", plain, stored);
    return 0;
}
"""


def test_no_term_reads_as_a_longer_row(tmp_path):
    text = open(os.path.join(ROOT, "farm_amd", "csrc", "hip", "intersection.hip")).read()
    mark = re.search(r"kRowLong = (0x[0-9a-f]+);", text).group(1)
    store = text[text.index("t[k] = ring.term("):text.index("t[0] = __hiloint2double(kRowLong")]
    guard = re.search(r"if \(.*\) t\[0\] = NAN;", store)
    src = tmp_path / "rows.c"
    src.write_text(SRC.replace("GUARD", guard.group(0).replace("t[0]", "t") if guard else ""))
    exe = str(tmp_path / "rows")
    subprocess.check_call(["gcc", "-O1", "-ffp-contract=off", str(src), "-o", exe, "-lm"])
    plain, stored = map(int, subprocess.check_output([exe, mark]).split())
    assert plain > 0  # such vertices exist
    assert stored == 0
