"""Device functions that take a node, the launch arguments or a descriptor by
reference are forced inline.  One that is called instead gets the object's
address: the object then lives in scratch memory and every pointer in it is
loaded as a generic one (see struct Node in csrc/vc_kernels.hip)."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallel-vertex-cover-algorithms-on-gpus_amd", "csrc")


def _device_functions():
    """(file, head up to the name, parameter list) of every device function."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"__device__([^;{}()]*)\(([^{};]*)\)\s*(?:const\s*)?\{", text):
            yield os.path.basename(path), m.group(1).strip(), m.group(2)


def test_functions_on_kernel_objects_are_inlined():
    seen, called = 0, []
    for name, head, params in _device_functions():
        if not re.search(r"\b(?:N|NodeT|SolveArgs|GDesc|BitsWorker|BitsLds|Cands)\s*&", params):
            continue
        seen += 1
        if "__forceinline__" not in head:
            called.append(f"{name}: {head}")
    assert seen >= 30, seen
    assert not called, called
