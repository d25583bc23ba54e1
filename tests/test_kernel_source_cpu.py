"""What the kernels' source must keep to that no compiler checks."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cellsim3d_amd", "csrc", "cs3d_kernels.hip")


def _functions(text):
    """(heading, body) of every function on file level: what precedes a brace at the start
    of an unindented declaration, up to the closing brace in the first column."""
    for m in re.finditer(r"^(?!namespace|struct|union|enum|constexpr|typedef|//|#|\})([^\n;{}]*(?:\n[^\n;{}]+)*\([^;{}]*\)\s*)\{\n(.*?)^\}", text,
                         re.M | re.S):
        yield m.group(1), m.group(2)


def test_kernel_arguments_are_read_in_kernels_only():
    """pool_late takes the kernel's argument segment, which is undefined in a called
    function: whatever reads it is a kernel or always inlined into one."""
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    found = [(h, b) for h, b in _functions(text) if re.search(r"pool_late\(\)|CS3D_LOOP_POOL\(", b)]
    names = [re.search(r"(\w+)\s*\([^()]*(?:\([^()]*\)[^()]*)*\)\s*$", h).group(1) for h, _ in found]
    assert {"k_integrate", "k_con_dis", "k_dis_post", "k_search", "divide_system"} <= set(names), names
    for name, (h, _) in zip(names, found):
        assert "__global__" in h or "__forceinline__" in h, name
        assert "noinline" not in h, name
