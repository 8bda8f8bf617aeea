"""Calls that use scratch for speed alone go on without it where the device has no memory left: the same results, no error.  A library
loaded in front of the HIP runtime refuses the allocations, in a process of its own and on a stream that has no scratch yet."""
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

REFUSE = r"""
#include <stddef.h>
static int (*real)(void**, size_t); static int refused = -1;
void refuse_real(void* f) { real = (int (*)(void**, size_t))f; }
void refuse(int on) { refused = on ? 0 : -1; }
int refusals(void) { return refused; }
int hipMalloc(void** p, size_t n) { if (refused >= 0) { refused++; *p = 0; return 2; } return real(p, n); }   /* hipErrorOutOfMemory */
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import torch
hip = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line)
shim.refuse_real(ctypes.cast(ctypes.CDLL(hip).hipMalloc, ctypes.c_void_p))
from sortnet_amd import ext
g = torch.Generator().manual_seed(1)
data = lambda *s: torch.randn(*s, generator=g).cuda()
out = lambda *s, t=torch.float32: torch.full(s, 7, device="cuda", dtype=t)
pos = lambda *s: out(*s, t=torch.int32)
calls = {}

x, w, gy = data(256, 512, 1), data(512, 512), data(256, 512, 1)
y = out(256, 512, 1)
ext.norm_dist_forward(x, w, y, 1, 8.0)
calls["l-p gradients"] = (lambda o, x=x, w=w, gy=gy, y=y: ext.norm_dist_backward_input_weight(gy, x, w, y, *o, 1, 8.0), [out(256, 512, 1), out(512, 512)])
xs, wc = data(80, 27, 1024), data(64, 27)
calls["convolution"] = (lambda o: ext.inf_dist_forward_nograd(xs, wc, *o, 1), [out(80, 64, 1024)])
calls["convolution, positions"] = (lambda o: ext.inf_dist_forward(xs, wc, *o, 1), [out(80, 64, 1024), pos(80, 64, 1024)])
xp, wp = data(128, 32, 1024), data(64, 32)
calls["convolution, l-p"] = (lambda o: ext.norm_dist_forward(xp, wp, *o, 1, 8.0), [out(128, 64, 1024)])
xo, wo = data(128, 1306, 1) * 0.05, data(1306, 1306)
calls["sort"] = (lambda o: ext.sort_neuron_forward_nograd(xo, wo, *o, 1, 0.75, 10), [out(128, 1306, 1)])
calls["sort, positions"] = (lambda o: ext.sort_neuron_forward(xo, wo, *o, 1, 0.75, 10), [out(128, 1306, 1), pos(10, 128, 1306, 1)])
lo, up = xo - 0.03, xo + 0.03
calls["sort, interval"] = (lambda o: ext.bound_sort_neuron_forward(lo, up, wo, *o, 1, 0.75, 10), [out(128, 1306, 1), out(128, 1306, 1)])
xb, wb = data(1024, 223, 1), data(1024, 223)
ub = xb + 0.1
calls["interval"] = (lambda o: ext.bound_inf_dist_forward_nograd(xb, ub, wb, *o, 1), [out(1024, 1024, 1), out(1024, 1024, 1)])
calls["interval, positions"] = (lambda o: ext.bound_inf_dist_forward(xb, ub, wb, *o, 1),
                                [out(1024, 1024, 1), out(1024, 1024, 1), pos(1024, 1024, 1), pos(1024, 1024, 1)])
calls["mask"] = (lambda o: ext.masked_inf_dist_forward(xb, wb, *o, None, 1, 0.3, 5, ext.MASK_FACTORED), [out(1024, 1024, 1)])
calls["mask, positions"] = (lambda o: ext.masked_inf_dist_forward(xb, wb, *o, 1, 0.3, 5, ext.MASK_FACTORED), [out(1024, 1024, 1), pos(1024, 1024, 1)])

for name, (fn, want) in calls.items():
    got = [torch.empty_like(t) for t in want]
    fn(want)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        for t in got:
            t.fill_(7)
        torch.cuda.synchronize()
        shim.refuse(1)
        try:
            fn(got)
            error = None
        except RuntimeError as e:
            error = e
        refused = shim.refusals()
        shim.refuse(0)
        torch.cuda.synchronize()
    if error is None and refused > 0:
        for a, b in zip(got, want):
            if "l-p" in name:
                torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5 * float(b.abs().max()))
            else:
                assert torch.equal(a, b), name
    print(name, "|", refused, "|", "ok" if error is None else error, flush=True)
"""


def test_short_of_memory(tmp_path):
    src, lib = tmp_path / "refuse.c", tmp_path / "refuse.so"
    src.write_text(REFUSE)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)])
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = [line.split(" | ") for line in r.stdout.splitlines() if " | " in line]
    assert len(lines) == 11 and all(int(refused) > 0 for _, refused, _ in lines), r.stdout   # (every one asks for scratch)
    assert all(result == "ok" for _, _, result in lines), r.stdout
