"""What the library does on the host, on a HIP runtime without a device (fake_hip.cpp): kernels are only named, and a
launch can be refused.  Each case runs in a process of its own, where that runtime stands in front of the real one."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PREAMBLE = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_launched.restype = ctypes.c_char_p
import numpy as np
from forja_amd import programs
from forja_amd.core import BackendError, CommandList, DType, Op
from forja_amd.hip_backend import HipBackend, load_library
hip = HipBackend(0)

def launched():
    names = fake.fake_launched().decode().split()
    fake.fake_forget()
    return names

def refuse(part):
    fake.fake_refuse(part.encode())
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    library = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", library], check=True)

    def run(body):
        script = PREAMBLE.format(root=ROOT, fake=library) + body
        result = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120)
        assert result.returncode == 0, result.stdout + result.stderr
    return run


def test_an_error_that_stood_before_a_call_is_not_its_own(fake):
    """A HIP call that failed elsewhere in the program leaves its error until someone asks."""
    fake("""
t = hip.alloc(DType.U32, (4,))
for call in (lambda: hip.write_array(t, np.arange(4, dtype=np.uint32)),
             lambda: hip.submit(CommandList()).wait(),
             lambda: hip.submit_static(CommandList())):
    fake.fake_fail()
    call()
assert np.frombuffer(hip.read_buffer_range(t.buffer, 0, 16), np.uint32).tolist() == [0, 1, 2, 3]
""")


def test_a_refused_move_is_noticed(fake):
    """Bytes read are the buffer's, and a submission's error records are looked at, also where the kernel that moves
    them is refused.  A gather that is refused fails the read, a dispatch the submission."""
    fake("""
t = hip.alloc(DType.U32, (64,))
values = np.arange(64, dtype=np.uint32)
for first in (0, 100):
    refuse("" if first == 0 else "move_bytes")
    hip.write_array(t, values + first)
    assert np.frombuffer(hip.read_buffer_range(t.buffer, 0, 256), np.uint32).tolist() == (values + first).tolist()
    hip.submit(CommandList()).wait()
    assert fake.fake_standing() == 0
copies = CommandList()
copies.dispatch(Op.copy(), [t], hip.alloc(DType.U32, (64,)))
for part, call in (("copy", lambda: hip.read(t)), ("copy", lambda: hip.submit(copies).wait()),
                   ("kernel", lambda: hip.submit(copies).wait())):
    refuse(part)
    try:
        call()
        raise SystemExit("a refused kernel has not been noticed")
    except BackendError:
        pass
""")


def test_which_reads_and_writes_a_kernel_moves(fake):
    """Up to 64 KiB, in the widest pieces that address and length allow; the copies of the runtime beyond."""
    fake("""
t = hip.alloc(DType.U32, (1 << 15,))
expected = bytearray(hip.read_buffer_range(t.buffer, 0, 1 << 17))
lib, rng = load_library(), np.random.default_rng(3)
widths = {16: "15HIP_vector_type", 4: "Ij", 1: "Ih"}
for first, length in ((0, 16), (16, 4080), (4, 20), (32, 36), (1, 16), (16, 3), (0, 16384), (4, 16380), (7, 16377), (0, 16385),
                      (8, 16388), (4, 65536), (0, 65537), (12, 100000)):
    data = rng.bytes(length)
    hip.synchronize()
    launched()
    assert lib.fh_write(hip._handle, t.buffer, first, data, length) == 0
    wrote = launched()
    expected[first:first + length] = data
    assert hip.read_buffer_range(t.buffer, first, first + length) == data
    read = launched()
    width = next(w for w in widths if (first | length) % w == 0)
    for names in (wrote, read):
        assert len(names) == (length <= 65536), (first, length, names)
        assert all(widths[width] in name and "move_bytes_kernel" in name for name in names), (first, length, names)
assert hip.read_buffer_range(t.buffer, 0, 1 << 17) == bytes(expected)
""")


@pytest.mark.parametrize("rows,n,k,form,expected", [
    # the normalisation in front: K up to 1024 ..
    (1, 6144, 1024, "norm", [2]), (16, 4096, 1024, "norm", [2]), (32, 4096, 768, "norm", [2]), (33, 4096, 1024, "norm", [1, 1]),
    (8, 5120, 2048, "norm", [1, 1]), (1, 2560, 1536, "res", [1, 1]),
    # .. with the residual sum over one row tile where a compute unit has one workgroup, rows are few or batches many
    (16, 4096, 768, "res", [2]), (16, 8192, 512, "res", [2]), (17, 4096, 768, "res", [1, 1]), (32, 1024, 512, "res", [2]),
    (4, 4160, 1024, "res", [2]), (5, 4160, 1024, "res", [1, 1]), (16, 8192, 1024, "res", [1, 1]), (16, 8256, 1024, "res", [2]),
    (16, 16384, 1024, "res", [2]), (8, 16448, 1024, "res", [2]), (9, 16448, 1024, "res", [1, 1]), (16, 65536, 1024, "res", [2]),
    # silu behind: wherever the kernel takes the product
    (16, 6144, 1024, "res-silu", [3]), (32, 6144, 1024, "norm-silu", [3]), (17, 6144, 1024, "res-silu", [1, 2]),
    (17, 6144, 512, "res-silu", [3]), (8, 6144, 2048, "norm-silu", [1, 2]), (32, 4096, 1536, "silu", [2]),
    (33, 6144, 1024, "res-silu", [1, 1, 1]), (4, 6144, 3072, "norm-silu", [1, 1, 1]), (4, 1008, 1024, "norm-silu", [1, 1, 1]),
    # not the rows the product reads, or not the halves of what it makes
    (4, 4096, 1024, "other-rows", [1, 1]), (4, 4096, 1024, "norm-other-halves", [2, 1])])
def test_which_row_programs_a_dense_product_takes_in(fake, rows, n, k, form, expected):
    """Dispatches of a joined group share one entry of the profile."""
    fake(f"""
rows, n, k, form, expected = {rows}, {n}, {k}, {form!r}, {expected}
x, u, normed, added, other = (hip.alloc(DType.BF16, (rows, k)) for _ in range(5))
w = hip.alloc(DType.BF16, (k,)).broadcast((rows, k))
weights = [hip.alloc(DType.U32, (n, k // 8)), *(hip.alloc(DType.BF16, (n, k // 64)) for _ in range(2))]
out, activated = hip.alloc(DType.BF16, (rows, n)), hip.alloc(DType.BF16, (rows, n // 2))
commands = CommandList()
if "res" in form:
    commands.dispatch_kernel(hip.prepare_program(programs.residual_norm_rows(1e-6)), [x, u, w], [added, normed])
elif form != "silu":
    commands.dispatch_kernel(hip.prepare_program(programs.rms_norm_rows(1e-6)), [x, w], [normed])
commands.dispatch(Op.quant_matmul(4, 64), [other if form == "other-rows" else normed, *weights], out)
if "silu" in form or "halves" in form:
    halves = [out.narrow(1, 0, n // 2), out.narrow(1, n // 2, n // 2)]
    commands.dispatch_kernel(hip.prepare_program(programs.silu_mul_elements()), halves if "silu" in form else halves[::-1], [activated])
submission = hip.submit_profiled(commands)
submission.wait()
got = [entry[1] for entry in submission.profile()]
assert got == expected, got
""")


def test_a_product_joined_with_its_normalisation_is_timed_as_a_product(fake):
    fake("""
x, normed, out = (hip.alloc(DType.BF16, (4, 1024)) for _ in range(3))
weights = [hip.alloc(DType.U32, (1024, 128)), *(hip.alloc(DType.BF16, (1024, 16)) for _ in range(2))]
commands = CommandList()
commands.dispatch_kernel(hip.prepare_program(programs.rms_norm_rows(1e-6)), [x, hip.alloc(DType.BF16, (1024,)).broadcast((4, 1024))], [normed])
commands.dispatch(Op.quant_matmul(4, 64), [normed, *weights], out)
hip.profile_enable(2)
hip.submit(commands).wait()
assert [hip.profile_read(kernel_class)[1] for kernel_class in (0, 1)] == [0, 1]   # other, products
""")


@pytest.mark.parametrize("lanes,pad,placed", [(1, 0, True), (4, 4, True), (4, 2, False), (128, 0, True), (129, 0, False)])
def test_who_places_the_lanes_rows(fake, lanes, pad, placed):
    """The merge where the destinations are aligned to four elements and one launch takes the lanes, else a scatter."""
    fake(f"""
lanes, pad, placed = {lanes}, {pad}, {placed}
from tests.test_lane_fusion_gpu import LaneBatch
batch = LaneBatch(hip, [5 + lane % 7 for lane in range(lanes)], 8, 2, 16, seed=1)
width = 8 * 128
target = hip.alloc(DType.BF16, (lanes, width + pad))
commands = CommandList()
for lane in range(lanes):
    row = hip.alloc(DType.BF16, (1, 8, 128))
    commands.dispatch_many(Op.paged_sdpa_append(0.09, 5 + lane % 7, 16),
                           [batch.q.narrow(0, lane, 1).permute([1, 0, 2]), batch.k.narrow(0, lane, 1),
                            batch.v.narrow(0, lane, 1), batch.tables[lane], batch.generations],
                           [row.permute([1, 0, 2]), *batch.pools[0]])
    commands.dispatch(Op.copy(), [row.reshape((1, width))], target.narrow(0, lane, 1).narrow(1, 0, width))
launched()
hip.submit(commands).wait()
assert hip.fusion_stats() == (1, 2 * lanes)
names = launched()
assert sum("ragged_reduce_kernelILb1" in name for name in names) == placed, names
assert any("scatter_lane_rows" in name for name in names) == (not placed), names
""")
