"""
A context belongs to one device, its caller's thread may have another one selected: a kernel launched on a stream of a
device that is not selected is refused. Every entry of the library that launches kernels selects the context's device
before it does. One GPU cannot show this, so the library's source is read: each function of the C interface whose body
launches a kernel, by itself or through a helper, must call hipSetDevice(ctx->device) first.
"""

import os
import re

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ionization_amd", "csrc", "engine.hip")


def _functions(text):
    """(name, body) of every function defined at the start of a line."""
    for m in re.finditer(r"^(?!static_assert|struct|using|namespace)[A-Za-z_][\w:<>*& ]*?\b(\w+)\((?:[^;{}]|\{\})*\)\s*\{", text, re.M):
        depth, i = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(text[i], 0)
            i += 1
        yield m.group(1), text[m.end():i]


def test_entries_that_launch_kernels_select_the_device():
    with open(SOURCE) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    bodies = dict(_functions(text))
    assert {"tdse_run", "tdse_tdma_batched", "tdse_materialize", "move_natural", "upload_state"} <= set(bodies)
    launches = {name for name, body in bodies.items() if "hipLaunchKernelGGL" in body}
    while True:
        more = {name for name, body in bodies.items() if name not in launches and any(
            re.search(rf"\b{callee}\s*(<[^;()]*>)?\(", body) for callee in launches)}
        if not more:
            break
        launches |= more
    entries = {name for name in launches if name.startswith("tdse_")}
    assert {"tdse_run", "tdse_tdma", "tdse_tdma_batched_noalloc", "tdse_upload_g", "tdse_download_g", "tdse_copy_probe",
            "tdse_materialize"} <= entries

    def selects(name):
        """hipSetDevice in the body before any launch, or only calls of functions that do so."""
        body = bodies[name]
        first = min([m.start() for callee in launches for m in re.finditer(rf"\b{callee}\s*(<[^;()]*>)?\(", body)]
                    + [m.start() for m in re.finditer("hipLaunchKernelGGL", body)])
        if 0 <= body.find("hipSetDevice(ctx->device)") < first:
            return True
        callees = [c for c in launches if re.search(rf"\b{c}\s*(<[^;()]*>)?\(", body)]
        return "hipLaunchKernelGGL" not in body and bool(callees) and all(selects(c) for c in callees)

    assert [name for name in sorted(entries) if not selects(name)] == []
