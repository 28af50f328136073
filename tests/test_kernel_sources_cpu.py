"""What the kernels' sources have to state whatever the present compiler makes of them (no GPU needed)."""
import os
import re

import pytest

HIPQ = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nart_amd", "csrc", "hipq")
LOAD, BARRIER = "__builtin_amdgcn_global_load_lds(", re.compile(r"__syncthreads\(\)|__builtin_amdgcn_s_barrier\(\)")
WAIT = re.compile(r"wait_vmcnt<[^;]*>\(\);|__builtin_amdgcn_s_waitcnt\(0\);")


def kernels():
    for f in sorted(os.listdir(HIPQ)):
        if f.endswith(".hip"):
            with open(os.path.join(HIPQ, f)) as src:
                text = re.sub(r"//[^\n]*", "", src.read())
            for m in re.finditer(r"__global__[^;{]*?(conv\w+_kernel)\(", text):
                start = depth = text.index("{", m.end())
                depth, end = 1, start + 1
                while depth:
                    depth += {"{": 1, "}": -1}.get(text[end], 0)
                    end += 1
                body = text[start:end]
                if LOAD in body:
                    yield pytest.param(body, id=m.group(1))


@pytest.mark.parametrize("body", kernels())
def test_loads_into_lds_are_waited_for_before_the_barrier(body):
    """The load unit writes LDS behind the compiler's back: a barrier alone orders nothing of it.  Between a kernel's first loads and the
    barrier in front of the reads the wait for them stands on every path: at the barrier's own nesting, or in both branches of an if."""
    at = body.index(LOAD)
    barrier = BARRIER.search(body, at)
    nesting = lambda i: body.count("{", 0, i) - body.count("}", 0, i)
    # an if without braces adds no nesting: the line in front of such a wait ends with its condition
    conditional = lambda i: re.search(r"(?:if \(.*\)|else)\s*$", body[:i].rstrip(" ")) is not None
    waits = [m.start() for m in WAIT.finditer(body, at, barrier.start())]
    always = [i for i in waits if nesting(i) <= nesting(barrier.start()) and not conditional(i)]
    both = [i for i in waits if re.search(r"else\s*$", body[:i])]
    assert always or both, "no wait on every path to the barrier"
