"""Kernels with written-out barriers: an s_barrier instruction waits for nothing, so
whatever a wave still has to read from LDS must have been waited for in front of it where
the buffer is filled again behind it.  Read from the gfx950 assembly of the sources."""
import os
import re
import subprocess

import pytest

from muxserve_amd import build

WAIT = re.compile(r"lgkmcnt\((\d+)\)")


def _functions(source):
    flags = [f for f in build.HIP_FLAGS if f not in ("-shared", "-fPIC")]
    text = subprocess.run([build.HIPCC, *flags, "-w", f"-I{build.INCLUDE}", f"-I{os.path.join(build.CSRC, 'hip')}", "-S",
                           "--offload-device-only", os.path.join(build.CSRC, "hip", source), "-o", "-"],
                          check=True, capture_output=True, text=True).stdout
    name, body = None, []
    for line in text.splitlines():
        code = line.split(";")[0].strip()
        if re.match(r"_ZN?\w+:$", code):
            name, body = code[:-1], []
        elif code.startswith(".Lfunc_end") and name:
            yield name, body
            name = None
        elif name and code and not code.startswith("."):
            body.append(code)
        elif name and re.match(r"\.LBB\w+:", code):
            body.append(code)


def _reads_left_at_barriers(body):
    """Per s_barrier, the most LDS reads (in order of issue, as the hardware counts them)
    that may not have arrived, over all paths to it."""
    labels = {code[:-1]: i for i, code in enumerate(body) if code.endswith(":")}
    best, left, work = {}, {}, [(0, 0)]
    while work:
        i, n = work.pop()
        while i < len(body) and best.get(i, -1) < n:
            best[i] = n
            code = body[i]
            op = code.split()[0]
            if op.startswith(("ds_read", "ds_load")):
                n = min(n + 1, 64)
            elif op.startswith("s_waitcnt") and WAIT.search(code):
                n = min(n, int(WAIT.search(code).group(1)))
            elif op == "s_barrier":
                left[i] = n
            if op.startswith("s_cbranch"):
                work.append((labels[code.split()[1]], n))
            elif op == "s_branch":
                i = labels[code.split()[1]]
                continue
            elif op == "s_endpgm":
                break
            i += 1
    return left


@pytest.mark.parametrize("source,kernels,count", [("sampler.hip", "lm_head_argmax_wide_kernel", 8),
                                                  ("prefill.hip", "prefill_", 10), ("model_ops.hip", "rms_norm_kernel", 16)])
def test_no_lds_read_is_outstanding_at_a_barrier(source, kernels, count):
    seen = 0
    for name, body in _functions(source):
        if kernels not in name:
            continue
        left = _reads_left_at_barriers(body).values()      # (workgroups of one wave have no barrier)
        assert not any(left), f"{name}: LDS reads outstanding at its barriers {sorted(left)}"
        seen += 1
    assert seen == count
