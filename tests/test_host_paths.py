"""The host side of the GEMM entry points without a GPU: which kernels a call
launches and which library buffers they get, on a recording stand-in for the
HIP runtime (tests/cpp/fake_hip.cpp) -- where an allocation fails, where the
stream captures a graph, and on several streams.  Each case runs in a process
of its own, since libmiq.so there binds to the stand-in."""
import os
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(REPO, "tests", "cpp", "fake_hip.cpp")

PRELUDE = r'''
import ctypes, importlib.util, os, re, sys
repo, fake_path = sys.argv[1:3]
fake = ctypes.CDLL(fake_path, mode=ctypes.RTLD_GLOBAL)
fake.fake_name.restype = ctypes.c_char_p
fake.fake_buffer.restype = fake.fake_allocated.restype = ctypes.c_uint64
fake.fake_malloc_limit.argtypes = [ctypes.c_size_t]
spec = importlib.util.spec_from_file_location("miq_host", os.path.join(repo, "sycl-infer_amd", "__init__.py"))
miq = importlib.util.module_from_spec(spec)
sys.modules["miq_host"] = miq
spec.loader.exec_module(miq)
lib = miq.lib()
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
OK, UNSUPPORTED, EHIP = 0, 1, -2
NO_LIMIT = 2**64 - 1

def seg(qt, n, k, tb, i=0):
    a = 0x100000000 + (i << 34)  # never read
    s = miq.Seg()
    s.w, s.type, s.K, s.n_rows, s.out, s.out_stride, s.alpha = a, qt, k, n, a + (1 << 32), n, 1.0
    s.x, s.x_stride = 0x4000000000, k
    s.x8, s.xmeta, s.xsumq = 0x4100000000, 0x4200000000, 0x4300000000
    return s

def run(fn, segs, tb, stream=0):
    """(status, kernel names, library buffers of each launch)"""
    fake.fake_reset()
    segs = segs if isinstance(segs, list) else [segs]
    f = getattr(lib, "miq_" + fn)
    if fn.endswith("multi"):
        rc = f(stream, (miq.Seg * len(segs))(*segs), len(segs), tb)
    else:
        rc = f(stream, ctypes.byref(segs[0]), tb)
    names, bufs = [], []
    for i in range(fake.fake_launches()):
        name = re.search(r"miq(?:12_GLOBAL__N_1)?\d+([a-z]\w*?_kernel)", fake.fake_name(i).decode()).group(1)
        if name != "zero_u32_kernel":  # clears new counters
            names.append(name)
            bufs.append([b for b in (fake.fake_buffer(i, k) for k in range(16)) if b])
    return rc, names, bufs

def sliced(n, tb):
    """whether the last launch, of the int8 tiled GEMM, has more workgroups than tiles (of 128 rows x 64 tokens)"""
    t = -(-n // 128) * -(-tb // 64)
    return fake.fake_blocks(fake.fake_launches() - 1) > -(-t // 8) * 8
'''


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", SRC,
                    "-o", lib], check=True, capture_output=True)

    def run(body, **env):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, REPO, lib], capture_output=True, text=True, timeout=60,
                           env={**os.environ, **env})
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_stand_in_records_launches(host):
    """one token, 16 tokens and a prefill batch: the GEMV, the 16-token kernel, pre-pass and GEMM"""
    host(r"""
rc, names, bufs = run("i8_gemm", seg(Q4_K, 4096, 4096, 1), 1)
assert rc == OK and len(names) == 1 and "gemv" in names[0], names
rc, names, bufs = run("i8_gemm", seg(Q4_K, 17408, 5120, 16), 16)
assert rc == OK and names == ["m16z_kernel"] and len(bufs[0]) == 2, (names, bufs)
rc, names, bufs = run("quant_gemm", seg(Q4_K, 17408, 5120, 512), 512)
assert rc == OK and names == ["pf_quant_kernel", "pf16_kernel"], (rc, names)
rc, names, bufs = run("i8_gemm", seg(Q8_0, 5120, 5120, 333), 333)
assert rc == OK and names == ["mfma32_kernel"] and len(bufs[0]) == 2 and sliced(5120, 333), (rc, names)
""")


def test_q80_prefill_scratch_is_the_streams_own(host):
    """Q8_0 prefill from 48 tokens on, on the sliced int8 GEMM and on the 16-token kernel (small matrices): the
    partials and counters of two streams are different buffers, those of one stream the same; a stream beyond the
    eighth, hipStreamPerThread, a capturing stream and miq_i8_gemm_noalloc get none and run the unsliced GEMM."""
    host(r"""
for fn in ("i8_gemm", "quant_gemm", "i8_gemv_multi"):
    for n, k, tb, kernel in ((5120, 5120, 333, "mfma32_kernel"), (1024, 5120, 64, "m16z_kernel")):
        s = [seg(Q8_0, n, k, tb)] if fn != "i8_gemv_multi" else [seg(Q8_0, n, k, tb, i) for i in range(2)]
        seen = {}
        for stream in (0, 0x5000, 0x6000, 0x5000, 0):
            rc, names, bufs = run(fn, s, tb, stream)
            assert rc == OK and names[-1] == kernel and len(bufs[-1]) == 2, (fn, rc, names, bufs)
            assert seen.setdefault(stream, bufs[-1]) == bufs[-1]
        assert len({b for v in seen.values() for b in v}) == 6, seen
        fake.fake_capturing(1)
        for stream in (0x5000, 0x7000):  # warmed up before or not
            rc, names, bufs = run(fn, s, tb, stream)
            assert rc == OK and names[-1] == "mfma32_kernel" and not bufs[-1] and not sliced(n, tb), (fn, names, bufs)
        fake.fake_capturing(0)
        rc, names, bufs = run(fn, s, tb, 2)
        assert rc == OK and names[-1] == "mfma32_kernel" and not bufs[-1] and not sliced(n, tb)
s = seg(Q8_0, 5120, 5120, 333)
rc, names, bufs = run("i8_gemm_noalloc", s, 333)
assert rc == OK and names == ["mfma32_kernel"] and not sliced(5120, 333)
got = [run("i8_gemm", s, 333, 0x10000 + 16 * i) for i in range(12)]
own = [g[2][0] for g in got if g[2][0]]
assert all(g[0] == OK for g in got) and len(own) == 5 and len({b[0] for b in own}) == 5, own
""")


def test_int8_prefill_of_k_quants_scratch_is_the_streams_own(host):
    """PREFILL_FP16=0: the K-quants on the int8 tiled GEMM, from 48 tokens on, as Q8_0"""
    host(r"""
bufs = [run("i8_gemm", seg(Q4_K, 5120, 5120, 200), 200, s) for s in (0x5000, 0x6000)]
assert all(b[0] == OK and b[1] == ["mfma32_kernel"] and len(b[2][0]) == 2 for b in bufs), bufs
assert not set(bufs[0][2][0]) & set(bufs[1][2][0])
""", MIQ_PREFILL_FP16="0")


def test_q80_sixteen_token_batches_share_the_device_scratch(host):
    """below 48 tokens Q8_0 keeps the device's scratch, also under a capture that it was warmed up for"""
    host(r"""
for n, k, tb, kernel in ((5120, 5120, 16, "m16z_kernel"), (5120, 5120, 40, "mfma32_kernel")):
    s = seg(Q8_0, n, k, tb)
    a, b = run("i8_gemm", s, tb, 0x5000), run("i8_gemm", s, tb, 0x6000)
    fake.fake_capturing(1)
    c = run("i8_gemm", s, tb, 0x7000)
    fake.fake_capturing(0)
    assert a == b == c and a[0] == OK and a[1] == [kernel] and len(a[2][0]) == 2, (a, b, c)
""")


def test_refused_multi_call_runs_nothing(host):
    """several 16-token segments under a capture whose scratch is too small for them together: refused as a whole,
    also where it would do for the first one alone"""
    host(r"""
first, second = seg(Q4_K, 640, 5120, 16), seg(Q4_K, 8192, 5120, 16, 1)
assert run("i8_gemv_multi", [first], 16)[0] == OK
fake.fake_capturing(1)
assert run("i8_gemv_multi", [first], 16)[0] == OK
rc, names, bufs = run("i8_gemv_multi", [first, second], 16)
assert rc == UNSUPPORTED and not names, (rc, names)
""")


def test_no_memory_for_scratch(host):
    """where an allocation fails, a call that can do with less still runs and reports no error: several prefill
    segments one by one, a batch below 48 tokens on the 16-token kernel, Q8_0 prefill unsliced"""
    host(r"""
MiB = 2**20
fake.fake_malloc_limit(1 * MiB)
rc, names, bufs = run("i8_gemm", seg(Q8_0, 5120, 5120, 333), 333)
assert rc == OK and names == ["mfma32_kernel"] and not bufs[0] and not sliced(5120, 333), (rc, names)
rc, names, bufs = run("i8_gemm", seg(Q8_0, 1024, 5120, 200), 200)
assert rc == OK and names == ["mfma32_kernel"] and not bufs[0] and not sliced(1024, 200), (rc, names)
fake.fake_malloc_limit(28 * MiB)
for fn in ("i8_gemm", "quant_gemm"):
    rc, names, bufs = run(fn, seg(Q4_K, 17408, 5120, 40), 40)
    assert rc == OK and names[-1] == "m16z_kernel", (rc, names)
fake.fake_malloc_limit(100 * MiB)
for fn in ("i8_gemv_multi", "quant_gemm_multi"):
    rc, names, bufs = run(fn, [seg(Q4_K, 17408, 5120, 512, i) for i in range(3)], 512)
    assert rc == OK and names.count("pf16_kernel") == 3, (rc, names)
fake.fake_malloc_limit(1 * MiB)
rc, names, bufs = run("i8_gemm", seg(Q4_K, 17408, 5120, 2048), 2048)
assert rc == EHIP and not names, (rc, names)
""")


def test_prefill_workspace_is_bounded(host):
    """eight prefill segments of 64 MiB of partial sums each: two launches over the same 256 MiB"""
    host(r"""
rc, names, bufs = run("quant_gemm_multi", [seg(Q4_K, 17408, 5120, 512, i) for i in range(8)], 512)
assert rc == OK and names == ["pf_quant_kernel", "pf16_kernel", "pf16_kernel"] and bufs[1] == bufs[2], (names, bufs)
assert fake.fake_allocated() < 1.25 * (256 + 16) * 2**20, fake.fake_allocated()
""")


def test_int8_prefill_forms(host):
    """the int8 tiled GEMM's instance without slices (one workgroup per tile) wherever a tile is not cut, else the
    sliced one (eight tiles' slices at a time)"""
    host(r"""
form = lambda: re.search(r"M32FormE(\d)", fake.fake_name(fake.fake_launches() - 1).decode()).group(1)
for n, k, tb, s in ((17408, 5120, 333, 1), (5120, 5120, 512, 1), (5120, 512, 100, 1), (5120, 5120, 333, 2), (5120, 5120, 48, 5)):
    rc, names, _ = run("i8_gemm", seg(Q8_0, n, k, tb), tb)
    t = -(-n // 128) * -(-tb // 64)
    assert rc == OK and names == ["mfma32_kernel"] and form() == ("0" if s == 1 else "1"), (n, k, tb, form())
    assert fake.fake_blocks(fake.fake_launches() - 1) == (t if s == 1 else -(-t // 8) * 8 * s), (n, k, tb)
""")


ROUTES = r"""
def kernel(qt, n, k, tb, fn="i8_gemm"):
    rc, names, _ = run(fn, seg(qt, n, k, tb), tb)
    assert rc == OK, rc
    return names[-1]
want = %r
for (qt, tb), k in want.items():
    assert kernel(qt, 17408, 5120, tb) == k + "_kernel", (qt, tb, kernel(qt, 17408, 5120, tb))
"""


@pytest.mark.parametrize("env,want", [
    ({}, {(12, 32): "m16z", (12, 33): "pf16", (8, 16): "m16z", (8, 17): "mfma32", (14, 48): "pf16"}),
    # the forced forms from 48 tokens on: below, no model says that they are the faster ones
    ({"MIQ_PREFILL_FP16": "0"}, {(12, 47): "m16z", (12, 48): "mfma32", (8, 47): "m16z", (8, 48): "mfma32", (14, 17): "m16z"}),
    ({"MIQ_PREFILL_FP16": "2"}, {(12, 47): "m16z", (12, 48): "pf16", (14, 47): "m16z", (14, 48): "pf16"}),
    ({"MIQ_PREFILL_FP16": "2", "MIQ_M32_MIN_TB": "17"}, {(12, 16): "m16z", (12, 17): "pf16"}),
    ({"MIQ_PREFILL_FP16": "0", "MIQ_M32_MIN_TB": "20"}, {(12, 19): "m16z", (12, 20): "mfma32"}),
    ({"MIQ_M32_MIN_TB": "100"}, {(12, 99): "m16z", (12, 100): "pf16", (8, 99): "m16z"}),
])
def test_smallest_prefill_batches(host, env, want):
    """the smallest batches of the prefill kernels by default and under the switches that force one"""
    host(ROUTES % want, **env)


def test_noalloc_smallest_prefill_batches(host):
    """miq_i8_gemm_noalloc keeps the 16-token kernel below 48 tokens, whatever miq_i8_gemm does there"""
    host(r"""
for qt, tb, want in ((Q4_K, 40, "m16z_kernel"), (Q8_0, 20, "m16z_kernel"), (Q8_0, 47, "m16z_kernel"), (Q8_0, 48, "mfma32_kernel")):
    rc, names, _ = run("i8_gemm_noalloc", seg(qt, 7168, 5120, tb), tb)
    assert rc == OK and names == [want], (qt, tb, rc, names)
""")


def test_capture_without_workspace(host):
    """a capturing stream and a prefill shape that was not run before: the 16-token kernel where it has its scratch
    and miq_i8_gemm_noalloc would use it too, else a refusal before anything runs; Q8_0 runs unsliced"""
    host(r"""
fake.fake_capturing(1)
small, large = seg(Q4_K, 17408, 5120, 40), seg(Q4_K, 17408, 5120, 512)
for fn in ("i8_gemm", "i8_gemv_multi"):
    assert run(fn, small, 40)[:2] == (UNSUPPORTED, []) and run(fn, large, 512)[:2] == (UNSUPPORTED, [])
rc, names, bufs = run("i8_gemm", seg(Q8_0, 5120, 5120, 40), 40)
assert rc == OK and names == ["mfma32_kernel"] and not bufs[0] and not sliced(5120, 40)
fake.fake_capturing(0)
miq.set_switch("M32_MIN_TB", 100)  # the 16-token kernel's scratch for 40 tokens, no workspace
assert run("i8_gemm", small, 40)[1] == ["m16z_kernel"]
miq.set_switch("M32_MIN_TB", miq.SWITCH_DEFAULT)
fake.fake_capturing(1)
for fn, pre in (("i8_gemm", []), ("i8_gemv_multi", []), ("quant_gemm", ["xq_kernel"]), ("quant_gemm_multi", ["xq_kernel"])):
    assert run(fn, small, 40)[:2] == (OK, pre + ["m16z_kernel"]), (fn, run(fn, small, 40))
assert run("i8_gemm", large, 512)[:2] == (UNSUPPORTED, [])
fake.fake_capturing(0)
assert run("quant_gemm", small, 40)[:2] == (OK, ["pf_quant_kernel", "pf16_kernel"])
fake.fake_capturing(1)
assert run("quant_gemm", small, 40)[:2] == (OK, ["pf_quant_kernel", "pf16_kernel"])
""")
