"""Properties of the kernels' sources that no run can show."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mpi_amd", "csrc")


def test_in_place_kernels_promise_no_separate_buffers():
    """The derivative kernels that hz_derivative_xy and hz_derivative_z run with
    the output in the input's place declare neither as __restrict__ (with it the
    compiler may move a load past a store, whatever today's one does)."""
    for source, kernel in (("fderiv.hip", "derivative_lines"), ("misc.hip", "derivative_kernel")):
        text = open(os.path.join(CSRC, source)).read()
        args = re.search(r"__global__[^;{]*?\b" + kernel + r"\((.*?)\)\s*\{", text, re.S).group(1)
        names = {name: qualifier for qualifier, name in
                 re.findall(r"\*\s*(__restrict__)?\s*(\w+)\s*(?:,|$)", args.replace("\n", " "))}
        assert not names["u"] and not names["out"], (source, args)
