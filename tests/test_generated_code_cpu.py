"""What the compiler makes of kernels whose speed turns on it, read from their gfx950 assembly; needs no GPU."""
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "causal-conv1d_amd"))


def _assembly(source, tmp_path):
    import build
    path = str(tmp_path / (source + ".s"))
    cmd = build.compile_command(source, path, ["--cuda-device-only", "-S"])
    cmd.remove("-c")
    subprocess.run(cmd, check=True, capture_output=True, timeout=300)
    return open(path).read()


def _kernels(text, name):
    """(mangled name, body) of every instance of a kernel."""
    found = re.findall(r"^(_ZN\S*%s\S+):.*?\n(.*?)^\.Lfunc_end" % name, text, re.S | re.M)
    assert found
    return found


def test_backward_tiles_do_not_wait_for_their_stores(tmp_path):
    """Behind the first store of dx nothing is left to wait for but stores: a vector-memory wait there holds a step up
    until the one in front has been written.  (A workgroup that adds up its own sums may add into memory at the end.)"""
    for name, body in _kernels(_assembly("cc1d_bwd_channelfirst_tile.hip", tmp_path), "bwd_channelfirst_tile_kernel"):
        steps = body[body.index("buffer_store_dwordx4"):]
        direct = re.search(r"tile_kernelILi\dELi\dELb[01]ELb([01])E", name).group(1) == "1"
        assert steps.count("s_waitcnt vmcnt") <= direct, name


def test_decode_of_a_few_tokens_keeps_eight_waves(tmp_path):
    """At most 64 registers, eight wavefronts a SIMD, with up to eight x rows in flight."""
    text = _assembly("cc1d_update.hip", tmp_path)
    counts = re.findall(r"\.name:\s+\S*update_tokens_kernel\S*.*?\.vgpr_count:\s+(\d+)", text, re.S)
    assert counts and all(int(n) <= 64 for n in counts), counts


def test_short_rows_ask_for_their_elements_at_once(tmp_path):
    """Channel-first forward, rows shorter than a vector: a lane's up to 4 (16-bit: 8) elements are its first loads, and none is
    waited for in front of the last."""
    for name, body in _kernels(_assembly("cc1d_fwd_channelfirst.hip", tmp_path), "fwd_channelfirst_short_kernelILi[0-2]ELi[2-4]ELb[01]ELi2E"):
        parts = body.split("global_load_")
        elements = 4 if "kernelILi0E" in name else 8
        assert not any("vmcnt" in part for part in parts[1:elements]), name
