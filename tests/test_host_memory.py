"""Who owns which device memory when, without a GPU: the library runs on a HIP runtime in host
memory (tests/native/fake_hip.cpp), in a process of its own, whose kernels do nothing."""
import json
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, json, sys
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL({lib!r})
lib.XGBGetLastError.restype = fake.fake_launches.restype = ctypes.c_char_p
fake.fake_live_bytes.restype = fake.fake_arg.restype = ctypes.c_uint64
fake.fake_synchronised.restype = ctypes.c_long
fake.fake_fail_after.argtypes = [ctypes.c_long]

def ok(status):
    assert status == 0, lib.XGBGetLastError().decode()

def device_array(shape, strides=None, device=0):
    ok(fake.hipSetDevice(device))
    n, p = 4, ctypes.c_void_p()
    for d in shape:
        n *= d
    ok(fake.hipMalloc(ctypes.byref(p), ctypes.c_size_t(n)))
    return json.dumps(dict(data=[p.value, True], shape=list(shape), strides=strides,
                           typestr="<f4", version=3, stream=1)).encode()

def matrix(rows, features, device=0):
    h = ctypes.c_void_p()
    a = device_array((rows, features), device=device)
    ok(lib.XGDMatrixCreateFromCudaArrayInterface(a, b'{{"missing": NaN}}', ctypes.byref(h)))
    return h
"""


@pytest.fixture(scope="session")
def host(dp, tmp_path_factory):
    """Runs code (after PRELUDE) on the host-memory runtime; returns what it printed as JSON."""
    fake = str(tmp_path_factory.mktemp("hip") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", fake,
                    os.path.join(HERE, "native", "fake_hip.cpp")], check=True)

    def run(code):
        text = PRELUDE.format(fake=fake, lib=dp.LIB_PATH) + textwrap.dedent(code)
        p = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True,
                           timeout=120)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout)

    return run


def _model(trees, splits):
    """Chains of `splits` splits: 2 * splits + 1 nodes a tree, one tree a round."""
    n = 2 * splits + 1
    left = [i + 1 if i % 2 == 0 and i < 2 * splits else -1 for i in range(n)]
    tree = {"left_children": left, "right_children": [c + 1 if c > 0 else -1 for c in left],
            "split_indices": [0] * n, "split_conditions": [0.5] * n, "default_left": [1] * n}
    return json.dumps({"learner": {
        "gradient_booster": {"model": {"iteration_indptr": list(range(trees + 1)),
                                       "tree_info": [0] * trees, "trees": [tree] * trees}},
        "learner_model_param": {"base_score": "[0]", "num_class": "0", "num_feature": "3"},
        "objective": {"name": "reg:squarederror"}}})


def test_a_failed_upload_leaves_the_last_forest(host):
    """A prediction whose forest finds no memory fails; the next one of the range before must
    not launch on what the failure left."""
    out = host(f"""
        text = {_model(40, 30)!r}.encode()
        b = ctypes.c_void_p()
        ok(lib.XGBoosterCreate(None, 0, ctypes.byref(b)))
        ok(lib.XGBoosterLoadModelFromBuffer(b, text, ctypes.c_uint64(len(text))))
        x = device_array((50, 3))
        shape, dim, res = ctypes.c_void_p(), ctypes.c_uint64(), ctypes.c_void_p()
        def predict(end):
            cfg = json.dumps(dict(type=1, training=False, iteration_begin=0, iteration_end=end,
                                  strict_shape=True, cache_id=0, missing=float("nan"))).encode()
            return lib.XGBoosterPredictFromCudaArray(b, x, cfg, None, ctypes.byref(shape),
                                                     ctypes.byref(dim), ctypes.byref(res))
        seen = []
        for fail in range(1, 12):  # the allocations that the larger forest is given
            ok(predict(2))
            before = [fake.fake_arg(i) for i in (5, 6)]
            fake.fake_fail_after(fail - 1)
            failed = predict(40)
            fake.fake_fail_after(-1)
            fake.fake_forget_launches()
            ok(predict(2))
            seen.append([failed, before, [fake.fake_arg(i) for i in (5, 6)]])
        print(json.dumps(seen))
    """)
    assert out[0][0] != 0  # without any allocation it cannot succeed
    for failed, before, after in out:
        assert all(before) and all(after)
        if failed:
            assert after == before


def test_a_matrix_waits_for_its_own_device(host):
    """Its blocks go back to the pool of the device they are on: that device must be idle, not
    the one that happens to be current."""
    out = host("""
        h = matrix(100, 5, device=1)
        ok(lib.XGDMatrixSetInfoFromInterface(h, b"label", device_array((100,), device=1)))
        label = device_array((100,), device=1)
        ok(fake.hipSetDevice(0))
        counts = [fake.fake_synchronised(1)]
        ok(lib.XGDMatrixSetInfoFromInterface(h, b"label", label))  # the old labels are given back
        counts.append(fake.fake_synchronised(1))
        ok(lib.XGDMatrixFree(h))
        counts.append(fake.fake_synchronised(1))
        now = ctypes.c_int()
        ok(fake.hipGetDevice(ctypes.byref(now)))
        h = matrix(10, 5, device=1)  # without labels: nothing of it is on device 0
        other = fake.fake_synchronised(0)
        ok(lib.XGDMatrixFree(h))
        print(json.dumps([counts, now.value, fake.fake_synchronised(0) - other]))
    """)
    (start, labels, freed), device, other = out
    assert start < labels < freed
    assert device == 0 and other == 0


POOL = """
lib._ZN2dp15device_pool_getEmPi.restype = lib._ZN2dp15pinned_pool_getEm.restype = ctypes.c_void_p
dev = ctypes.c_int()
def get(n, pinned=False):
    if pinned:
        return lib._ZN2dp15pinned_pool_getEm(ctypes.c_size_t(n))
    return lib._ZN2dp15device_pool_getEmPi(ctypes.c_size_t(n), ctypes.byref(dev))
def put(p, n, pinned=False):
    if pinned:
        lib._ZN2dp15pinned_pool_putEPvm(ctypes.c_void_p(p), ctypes.c_size_t(n))
    else:
        lib._ZN2dp15device_pool_putEPvmi(ctypes.c_void_p(p), ctypes.c_size_t(n), dev)
MB = 1 << 20
"""


@pytest.mark.parametrize("pinned,total,largest", [(False, 24 << 30, 12 << 30),
                                                  (True, 2 << 30, 512 << 20)])
def test_what_the_pool_keeps_is_bounded(host, pinned, total, largest):
    """Device memory up to 24 GiB; host memory, which is never much, far less."""
    out = host(POOL + f"""
kind, pinned = ({-1 if pinned else 0}, {pinned})
live = []
for block in ({total // 64}, {largest}, {largest} + MB):
    held = [get(block, pinned) for _ in range(70)] if block < MB * 512 else [get(block, pinned)]
    for p in held: put(p, block, pinned)
    live.append(fake.fake_live_bytes(kind))
print(json.dumps(live))
""")
    many, one, larger = out
    assert many == total  # 64 of 70 blocks stay
    assert one == total   # the largest evicts as much as it brings
    assert larger <= total  # a larger one is never kept


@pytest.mark.parametrize("size", [1, 256, 257, 1 << 20, (1 << 20) + 1, (9 << 30) + 1, 12 << 30,
                                  (12 << 30) + 1, (17 << 30) + 255])
def test_blocks_that_are_not_kept_are_not_rounded_up(host, size):
    """Kept blocks come in sizes that later ones can share, at most a sixteenth larger; a block
    too large to be kept takes 256-byte units, as the driver's own allocations do."""
    got = host(POOL + f"""
p = get({size})
print(json.dumps(fake.fake_live_bytes(0)))
""")
    assert size <= got and got % 256 == 0
    assert got <= (size + 255 if size <= 1 << 20 or size > 12 << 30 else size * 17 // 16)


def test_kept_memory_can_be_handed_back(host):
    """Freed matrices' blocks stay for the next ones until the program asks for them."""
    out = host("""
        h = matrix(1000, 50)
        second = matrix(10, 5, device=1)
        before = [fake.fake_live_bytes(d) for d in (0, 1)]
        ok(lib.XGDMatrixFree(h))
        freed = fake.fake_live_bytes(0)
        ok(lib.DPReleaseCachedMemory())
        after = [fake.fake_live_bytes(d) for d in (0, 1)]
        ok(lib.DPReleaseCachedMemory())
        print(json.dumps([before, freed, after]))
    """)
    before, freed, after = out
    assert freed == before[0]
    assert after[0] == 4 * 1000 * 50  # the program's own array
    assert 4 * 10 * 5 * 2 <= after[1] <= before[1]  # a live matrix keeps its copy


@pytest.mark.parametrize("rows,features", [(5000, 8), (5000, 40)])
@pytest.mark.parametrize("booster", [True, False])
def test_the_tuner_times_what_runs(host, rows, features, booster):
    """The booster's passes end in the reduce that also evaluates, the operators' in the reduce
    alone; the operators time the contiguous pass only."""
    names = host(f"""
        class Layout(ctypes.Structure):
            _fields_ = [("rows", ctypes.c_int64), ("features", ctypes.c_int32),
                        ("width", ctypes.c_int32), ("tiles", ctypes.c_int32),
                        ("missing", ctypes.c_int32), ("pairs", ctypes.c_uint64)]
        lay = Layout()
        ok(lib.dp_layout_init(ctypes.c_int64({rows}), {features}, 0, -1, ctypes.byref(lay)))
        p = ctypes.c_void_p()
        ok(fake.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 20)))
        tune = lib._ZN2dp15tune_dense_histERK13dp_bin_layoutPKhbiPKiP12ihipStream_tS4_
        tune.restype = ctypes.c_void_p
        tune(ctypes.byref(lay), p, ctypes.c_bool({booster}), 256, p, None, None)
        print(json.dumps([x.split(" ")[0] for x in fake.fake_launches().decode().split(";") if x]))
    """)
    assert any("reduce_evaluate_dense" in n for n in names) == booster
    assert any("hist_reduce" in n for n in names) != booster


@pytest.mark.parametrize("rows,features,blocks", [(20000, 65536, 1), (20000, 65537, 2),
                                                  (1 << 26, 256, 1), (1 << 26, 1025, 5),
                                                  (1 << 31, 300, 3)])
def test_the_sketch_takes_features_by_blocks(host, rows, features, blocks):
    """Its scratch is bounded: at most 2^16 features at once, and 2^34 values or 128 features."""
    sampled = host(f"""
        ws, p = ctypes.c_void_p(), ctypes.c_void_p()
        ok(lib.dp_workspace_create(ctypes.byref(ws)))
        ok(fake.hipMalloc(ctypes.byref(p), ctypes.c_size_t(4)))  # the kernels do not run
        n = {features}
        ptr, cuts = (ctypes.c_int32 * (n + 1))(), (ctypes.c_float * (n * 16))()
        mins, missing = (ctypes.c_float * n)(), ctypes.c_int32()
        lib.dp_sketch_cuts(ws, p, ctypes.c_int64({rows}), n, 16, ptr, cuts, mins,
                           ctypes.byref(missing), None)
        names = fake.fake_launches().decode().split(";")
        print(json.dumps(sum("sample_kernel" in x for x in names)))
    """)
    assert sampled == blocks
