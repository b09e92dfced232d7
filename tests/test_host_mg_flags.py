"""The convergence flag of the multigrid BiCGSTAB (cp_mg.hip) on the device: a kernel that writes it
does not read it, since its blocks, and the waves of one block, would see either value, and no kernel
of an iteration's second part, which is queued only while the flag is clear, tests it."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-cpfem_amd", "csrc", "cp_mg.hip")


def _kernels():
    """Name -> text of each __global__ function, comments left out."""
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    out = {}
    for m in re.finditer(r"__global__[^;{]*?\b(k_\w+)\s*\(", text):
        start = text.index("{", m.end())
        depth, i = 1, start + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[i], 0)
            i += 1
        out[m.group(1)] = text[m.start():i]
    return out


def test_a_kernel_that_sets_the_flag_does_not_read_it():
    setters = 0
    for name, body in _kernels().items():
        writes = re.findall(r"->done\s*=(?!=)", body)
        setters += bool(writes)
        if writes:
            assert len(re.findall(r"\bdone\b", body)) == len(writes), name
    assert setters == 2  # k_mgb_init2 and k_mgb_p


def test_only_the_smoothing_kernels_test_the_flag():
    readers = {name for name, body in _kernels().items() if re.search(r"\bdone\b(?!\s*=[^=])", body)}
    assert readers == {"k_mg_smooth", "k_mg_resid"}
