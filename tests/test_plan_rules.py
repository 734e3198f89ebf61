"""Host-side launch rules (katali-lab_amd/csrc/kq_plan.h), compiled with the
host compiler and run here; no device.

The rule that decides whether a layer may run as one of the
launches whose workgroups wait for each other (the XCD-sliced layer and its
stack): every one of its 256 workgroups must be resident at once, one per CU
of a 256-CU device, with the occupancy API reporting at least one block of
the kernel per CU (launch_moe_xcd and launch_moe_stack).

The wide down projection's plan: every shape that the layer's LDS rule admits
has one, on any CU count, within the LDS, its row index exact.

Kernel A's half units: where the busiest CU has less work with them."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "katali-lab_amd", "csrc")

DRIVER = r"""
#include <stdio.h>
#include "kq_plan.h"
int main() {
    struct { int cus, bpc; unsigned grid; } c[] = {
        {256, 1, 256}, {256, 2, 256}, {256, 0, 256}, {304, 1, 256}, {128, 2, 256}, {0, 4, 256}, {-1, 1, 256},
        {80, 1, 80}, {256, 1, 512}};
    for (unsigned i = 0; i < sizeof c / sizeof c[0]; i++) printf("%d\n", kq::xcd_coresident(c[i].cus, c[i].bpc, c[i].grid) ? 1 : 0);
    return 0;
}
"""


DOWN_DRIVER = r"""
#include <stdio.h>
#include "kq_plan.h"
// every shape of rows above four blocks that the layer's LDS rule admits
int main() {
    unsigned long n = 0, ragged = 0, packed = 0, bad = 0;
    for (unsigned cus : {20u, 32u, 38u, 64u, 80u, 228u, 256u, 304u})
        for (unsigned hidden : {256u, 512u, 1024u, 2048u, 4096u})
            for (unsigned nb = 5; nb <= 64; nb++)
                for (unsigned slots = 1; slots <= 17 && slots * nb * 352 + 2116 <= 163840; slots++)
                    for (int q6 = 0; q6 < 2; q6++) {
                        kq::DownPlan p;
                        const unsigned ipb = q6 ? 4 : 8, ffn = 256 * nb;
                        bool ok = kq::down_plan(q6, hidden, ffn, slots, cus, p);
                        n++;
                        if (!ok) { bad++; continue; }
                        const unsigned tile = 16 / ipb * 352, gaps = slots * ((nb * ipb + 15) / 16) * tile;
                        const unsigned h = p.pack ? (slots * nb * ipb + 15) / 16 * tile : gaps;
                        packed += p.pack;
                        if (p.pack && gaps + 4 * (slots + 17) < 100000) bad++;   // packed only near the limit
                        ok = p.lds <= 163840 && p.lds >= h + (p.rpw * slots + 17) * 4 && p.rpw >= 1 && p.rpw <= 64 * p.nw &&
                             p.nw >= 4 && p.nw <= 16 && p.S == (nb > 16 ? 64 : 4 * ipb) && p.N >= 1 && p.N <= (q6 ? 4 : 8);
                        for (unsigned pc = 0; pc < p.rpw * slots; pc++) ok = ok && pc * p.inv_rpw >> 20 == pc / p.rpw;
                        ragged += hidden % p.rpw != 0;
                        if (!ok) bad++;
                    }
    printf("%lu %lu %lu %lu\n", n, ragged, packed, bad);
    return 0;
}
"""


HALF_DRIVER = r"""
#include <stdio.h>
#include "kq_plan.h"
int main() {
    for (unsigned u = 8; u <= 1160; u++)
        if (kq::half_units(u, 256)) printf("%u\n", u);
    return 0;
}
"""


def run_driver(tmp_path, code):
    src = tmp_path / "plan.cpp"
    src.write_text(code)
    exe = tmp_path / "plan"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], capture_output=True,
                       text=True)
    if r.returncode:
        pytest.fail(r.stderr)
    return subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()


def test_down_plan(tmp_path):
    n, ragged, packed, bad = map(int, run_driver(tmp_path, DOWN_DRIVER))
    assert n > 10000 and ragged > 0 and 0 < packed < n // 10 and bad == 0


def test_coresident_rule(tmp_path):
    out = run_driver(tmp_path, DRIVER)
    # one per CU on exactly 256 CUs: yes; a kernel that fits no CU, another
    # CU count (the slot-to-XCD mapping needs 256), a grid above the CUs: no
    assert out == ["1", "1", "0", "0", "0", "0", "0", "1", "0"]


def test_half_units_rule(tmp_path):
    got = list(map(int, run_driver(tmp_path, HALF_DRIVER)))
    # whole workgroups of eight units, in the lower half of each round of CUs
    want = [u for u in range(8, 1161) if u % 8 == 0 and (0 < u % 256 <= 128)]
    assert got == want and 896 in got and 1056 in got and not any(896 < u <= 1024 for u in got)
