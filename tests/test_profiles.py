"""The measurement summaries under profiles/ say which tree they were taken at, and the one bench.py reads
numbers from (measured HBM traffic per GEMM launch) must have been taken with the GEMM kernels of this tree."""
import os
import re

from fastconv_amd import provenance

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROFILES = os.path.join(ROOT, "profiles")


def test_every_summary_names_its_command_and_the_tree_it_was_taken_at():
    names = sorted(n for n in os.listdir(PROFILES) if n.endswith((".txt", ".md")))
    assert names
    for n in names:
        path = os.path.join(PROFILES, n)
        assert provenance.parse(path) is not None, "%s has no provenance line" % n
        text = open(path).read()
        assert "rocprofv3" in text or "bench.py" in text or "conv_test" in text, "%s does not give its command" % n
        assert os.path.getsize(path) < 64 * 1024, "%s is not a short summary" % n


def test_digest_follows_the_sources():
    everything = provenance.digest()
    assert len(everything) == 16 and everything == provenance.digest()
    assert provenance.digest(["wino_gemm.hip"]) != provenance.digest(["implicit_gemm.hip"])
    changed = provenance.digest(["wino_gemm.hip"], read=lambda n: b"something else")
    assert changed != provenance.digest(["wino_gemm.hip"])


def test_traffic_summary_was_measured_on_the_gemm_kernels_of_this_tree():
    """When the sources of the GEMM kernels change, headers included, profiles/gemm_hbm_traffic_pmc.txt has to be taken again
    (its commands are in its header); until then bench.py reports roofline.traffic as null."""
    path = os.path.join(PROFILES, "gemm_hbm_traffic_pmc.txt")
    commit, _, sources_digest, sources = provenance.parse(path)
    assert sources and sources_digest
    # the files of the kernels it names, with the headers that they include
    text = {n: open(os.path.join(provenance.CSRC, n)).read() for n in os.listdir(provenance.CSRC) if n.endswith((".hip", ".h"))}
    kernels = set(re.findall(r"^traffic kernel=(\w+)", open(path).read(), re.M))
    need = {n for n in text for k in kernels if n.endswith(".hip") and re.search(r"__global__[^;{]*\b%s\(" % k, text[n])}
    assert len(kernels) >= 3 and len(need) == len(kernels)
    while True:
        more = {h for n in need for h in re.findall(r'#include "(\w+\.h)"', text[n]) if h in text} - need
        if not more:
            break
        need |= more
    assert need <= set(sources), sorted(need - set(sources))
    assert provenance.sources_current(path), (
        "%s changed since commit %s: measure the HBM traffic of the GEMM kernels again" % (", ".join(sources), commit))
