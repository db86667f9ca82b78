"""The XLA FFI handlers that check what the C ABI cannot (an operand's length and dtype),
compiled against a stub of XLA's API (tests/xla_stub: the real headers are not here) and
called on the host. Against XLA itself: parity unpinned."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_operands_of_other_lengths_and_dtypes_are_refused(tmp_path):
    exe = tmp_path / "handlers"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(HERE, "xla_stub"),
                    "-I", os.path.join(os.path.dirname(HERE), "include"), "-I", "/opt/rocm/include",
                    os.path.join(HERE, "xla_handlers.cc"), "-o", str(exe)], check=True)
    got = [[int(v) for v in line.split()]
           for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]
    ok, refused = 0, 1
    sorts, biases = got[:7], got[7:]
    # the code, the calls of the library, the weights' bytes, whether there is a list
    assert sorts[:2] == [[ok, 1, 2, 1], [ok, 1, 4, 0]]
    assert all(line[:2] == [refused, 0] for line in sorts[2:])
    assert biases[:2] == [[ok, 1, 0], [ok, 1, 1]]  # BUX_BF16, BUX_F32
    assert all(line[:2] == [refused, 0] for line in biases[2:])
