"""Which kernel, grid and arguments a launch takes, on the CPU: the kernel library
runs in a child process on a stand-in for the HIP runtime, which records the launches
instead of making them and can be told to refuse a device query."""
import json
import os
import random
import subprocess
import sys

import pytest

from ridge_amd import gemm as G

FAKE_HIP = r"""
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
typedef struct { uint32_t x, y, z; } dim3_t;
static struct { const void* fn; const char* name; } kernels[4096];
static int count, error;
static dim3_t grid, block;
static size_t shared;
static void* stream;

void** __hipRegisterFatBinary(const void* data) { static void* handle; (void)data; return &handle; }
void __hipUnregisterFatBinary(void** modules) { (void)modules; }
void __hipRegisterFunction(void** modules, const void* host, char* device, const char* name, unsigned limit,
                           void* tid, void* bid, dim3_t* b, dim3_t* g, int* w) {
    (void)modules; (void)device; (void)limit; (void)tid; (void)bid; (void)b; (void)g; (void)w;
    if (count < 4096) { kernels[count].fn = host; kernels[count++].name = name; }
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t n, void* s) {
    grid = g; block = b; shared = n; stream = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* n, void** s) {
    *g = grid; *b = block; *n = shared; *s = stream;
    return 0;
}
int hipLaunchKernel(const void* fn, dim3_t g, dim3_t b, void** args, size_t n, void* s) {
    const char* name = "";
    (void)n; (void)s;
    for (int i = 0; i < count; ++i)
        if (kernels[i].fn == fn) name = kernels[i].name;
    const int ints = strstr(name, "PingPong") ? 8 : strstr(name, "Persistent") ? 9 : strstr(name, "Small") ? 5 : 6;
    printf("{\"kernel\": \"%s\", \"grid\": %u, \"block\": %u, \"args\": [", name, g.x, b.x);
    for (int i = 0; i < ints; ++i) printf("%s%u", i ? ", " : "", *(uint32_t*)args[3 + i]);
    printf("]}\n");
    fflush(stdout);
    return 0;
}
static int refused(const char* what) {
    const char* names = getenv("FAKE_HIP_REFUSES");
    if (names == 0 || strstr(names, what) == 0) return 0;
    error = 101;
    return 1;
}
int hipGetDevice(int* device) { if (refused("hipGetDevice")) return 101; *device = 0; return 0; }
int hipDeviceGetAttribute(int* value, int attribute, int device) {
    (void)attribute; (void)device;
    if (refused("hipDeviceGetAttribute")) return 101;
    *value = 256;
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void* fn, int threads, size_t n) {
    (void)fn; (void)threads; (void)n;
    if (refused("hipOccupancy")) return 101;
    *blocks = 1;
    return 0;
}
int hipGetLastError(void) { const int e = error; error = 0; return e; }
"""

# Loads the stand-in first and globally, so that the library's references bind to it.
CHILD = r"""
import ctypes, json, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
L = ctypes.CDLL(sys.argv[2])
launch = getattr(L, sys.argv[3])
launch.argtypes = [ctypes.c_int] + [ctypes.c_void_p] * 3 + [ctypes.c_int] * 3 + [ctypes.c_void_p]
for call in json.load(sys.stdin):
    rc = launch(call[0], 4096, 4096, 4096, call[1], call[2], call[3], None)
    print(json.dumps({"rc": rc}), flush=True)
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    d = tmp_path_factory.mktemp("fake_hip")
    src, so = d / "fake_hip.c", d / "libfake_hip.so"
    src.write_text(FAKE_HIP)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    return str(so)


def launches(fake_hip, calls, refuses="", entry="ridge_gemm_launch"):
    """[(return code, the launches made)] of calls (variant index, M, N, K)."""
    env = dict(os.environ, FAKE_HIP_REFUSES=refuses)
    p = subprocess.run([sys.executable, "-c", CHILD, fake_hip, G.LIB_PATH, entry], input=json.dumps(calls),
                       env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
    out, made = [], []
    for line in p.stdout.splitlines():
        r = json.loads(line)
        if "rc" in r:
            out.append((r["rc"], made))
            made = []
        else:
            made.append(r)
    assert len(out) == len(calls)
    return out


def rows(schedule=None, **fields):
    return [v for v in G.variants() if (schedule is None or v.schedule == schedule) and
            all(getattr(v, k) == x for k, x in fields.items())]


def ping_pong_parts(launch):
    """(whole tiles, workgroups of parts, parts per tile) of a ping-pong launch."""
    whole, part_tiles, parts_and_phase = launch["args"][5:8]
    return whole, part_tiles, parts_and_phase & 0xff


# 130849 and 133153 tiles: 33 behind whole rounds of 256, which fit one round as
# quarters. The quarters have BK = 64, and their last B row starts 63 * N * 2 bytes
# into the tile: 32 bits hold that for the first N and not for the second.
@pytest.mark.parametrize("N,parts", [(33497344, 4), (34087168, 2)])
def test_parts_whose_b_offsets_pass_32_bits_are_not_taken(fake_hip, N, parts):
    wide = rows(1, BM=256, BN=256, BK=32)
    assert len(wide) == 8
    tiles = N // 256
    for v, (rc, made) in zip(wide, launches(fake_hip, [(v.index, 256, N, 64) for v in wide])):
        assert rc == 0 and len(made) == 1
        assert ping_pong_parts(made[0]) == (tiles - 33, 33 * parts, parts), v.label()
        # What the blocks address: BK rows of B (halves keep the row's 32).
        assert (64 if parts >= 4 else 32) * N < 2 ** 31


def test_c_above_64_mib_is_stored_non_temporally_but_for_a_single_32_deep_step(fake_hip):
    """The kernels' bool template argument (Lb1E): true above 64 MiB of C, where
    non-temporal stores are the faster ones; a ping-pong row's K of 32 is not."""
    for v in rows(0) + rows(1):
        shapes = [(8192, 4096, K) for K in (32, 64)] + [(8192, 6144, K) for K in (32, 64, 128)]
        shapes = [s for s in shapes if v.divides(*s)]
        for (M, N, K), (rc, made) in zip(shapes, launches(fake_hip, [(v.index,) + s for s in shapes])):
            assert rc == 0 and len(made) == 1
            nt = M * N * 2 > 64 << 20 and not (v.schedule == 1 and K < 64)
            assert ("ELb1E" in made[0]["kernel"]) == nt, (v.label(), M, N, K, made[0]["kernel"])


@pytest.mark.parametrize("query", ["hipGetDevice", "hipDeviceGetAttribute", "hipOccupancy"])
def test_a_launch_whose_device_query_fails_runs_its_own_tiles_and_succeeds(fake_hip, query):
    """Uniform and ping-pong rows only choose smaller blocks by the device's CUs: where
    those are not to be had, the launch is the whole grid of the row's tile, and the
    query's error is not reported as the launch's."""
    picked = rows(0) + rows(1)
    M, N, K = 1024, 1024, 128
    for v, (rc, made) in zip(picked, launches(fake_hip, [(v.index, M, N, K) for v in picked], query)):
        assert rc == 0 and len(made) == 1, v.label()
        if query != "hipOccupancy":
            assert made[0]["grid"] == (M // v.BM) * (N // v.BN), v.label()
            assert made[0]["block"] == v.threads, v.label()


@pytest.mark.parametrize("M,N,K,block", [(1024, 1024, 128, (64, 64)), (2048, 1024, 128, (64, 128)),
                                         (2048, 2048, 128, (128, 128)), (4096, 4096, 128, None),
                                         (1024, 1024, 96, None)])
def test_small_grids_run_one_kernel_per_block_whatever_the_row(fake_hip, M, N, K, block):
    """A uniform or persistent row's grid of at most 128 tiles on 256 CUs, in the
    smallest block whose workgroups fit one round: the same kernel for every row."""
    names = {}
    picked = [v for v in rows(0) + rows(2) if v.divides(M, N, K) and (v.BM, v.BN) != (64, 64)]
    for v, (rc, made) in zip(picked, launches(fake_hip, [(v.index, M, N, K) for v in picked])):
        assert rc == 0 and len(made) == 1
        tiles = (M // v.BM) * (N // v.BN)
        small = "SmallGrid" in made[0]["kernel"]
        assert small == (tiles <= 128 and block is not None), v.label()
        if small:
            assert made[0]["grid"] == (M // block[0]) * (N // block[1]), v.label()
            names.setdefault(made[0]["kernel"], []).append(v.index)
        elif v.schedule == 0:
            assert made[0]["grid"] == tiles, v.label()
    assert len(names) == (1 if block else 0), names


def _form_shapes(v):
    """Grids on every side of the rules on 256 CUs: tile counts around half a round and
    around a sixteenth, an eighth, a quarter and a half of a round, alone and behind
    whole rounds; K on and off the parts' 64; N beyond what their offsets hold."""
    rng = random.Random(v.index)
    counts = [1, 2, 3, 16, 17, 32, 33, 64, 65, 100, 127, 128, 129, 200, 256]
    shapes = []
    for n in counts + [256 + c for c in counts] + [1024 + c for c in counts]:
        m = rng.choice([d for d in range(1, n + 1) if n % d == 0])
        shapes.append((v.BM * m, v.BN * (n // m), v.BK * rng.choice([1, 2, 3, 8])))
    shapes += [(v.BM, v.BN * (130816 + c), 64) for c in (1, 16, 33, 65, 129)]
    shapes += [(v.BM, v.BN * (133120 + c), 64) for c in (1, 16, 33, 65, 129)]
    return [s for s in shapes if v.divides(*s)]


@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_launch_form_says_what_the_launch_runs(fake_hip, schedule):
    picked = [(v, s) for v in rows(schedule) for s in _form_shapes(v)]
    kinds = set()
    for (v, (M, N, K)), (rc, made) in zip(picked, launches(fake_hip, [(v.index,) + s for v, s in picked])):
        what = "%s on %dx%dx%d" % (v.label(), M, N, K)
        assert rc == 0 and len(made) == 1, what
        f, tiles = G.launch_form(v.index, M, N, K), (M // v.BM) * (N // v.BN)
        # Every output once, in blocks that fit one round, the shape and 32-bit offsets.
        assert f.ownTiles * v.BM * v.BN + f.partWorkgroups * f.partBM * f.partBN == M * N, what
        assert f.own == (f.partBM == 0) == (f.ownTiles == tiles), what
        if not f.own:
            assert f.partWorkgroups <= 256 and K % f.partBK == 0, what
            assert f.partBK * N < 2 ** 31 and f.partBM * K < 2 ** 31, what
            assert (f.partBM // f.partWM) * (f.partBN // f.partWN) * 64 == 512, what
        if schedule == 1:
            whole, part_workgroups, parts = ping_pong_parts(made[0])
            assert (whole, part_workgroups) == (f.ownTiles, f.partWorkgroups), what
            assert made[0]["grid"] == whole + part_workgroups and tiles == whole + part_workgroups // parts, what
        else:
            assert f.own == ("SmallGrid" not in made[0]["kernel"]) and f.ownTiles in (0, tiles), what
            want = f.partWorkgroups if not f.own else tiles if schedule == 0 else min(tiles, 256)
            assert made[0]["grid"] == want, what
        kinds.add((f.partBM, f.partBN, f.partBK))
    assert len(kinds) == {0: 4, 1: 5, 2: 4}[schedule], kinds


@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_launch_own_tile_runs_the_rows_tile_on_every_grid(fake_hip, schedule):
    picked = [(v, s) for v in rows(schedule) for s in _form_shapes(v)]
    calls = [(v.index,) + s for v, s in picked]
    for (v, (M, N, K)), (rc, made) in zip(picked, launches(fake_hip, calls, entry="ridge_gemm_launch_own_tile")):
        tiles = (M // v.BM) * (N // v.BN)
        assert rc == 0 and len(made) == 1 and "SmallGrid" not in made[0]["kernel"]
        assert made[0]["grid"] == (min(tiles, 256) if schedule == 2 else tiles)
        assert made[0]["block"] == v.threads
        if schedule == 1:
            assert ping_pong_parts(made[0]) == (tiles, 0, 1)


def test_launch_form_refuses_what_a_launch_refuses():
    for args in ((-1, 256, 256, 64), (0, 255, 256, 64), (0, 256, 256, 64, 0), (G.num_variants(), 256, 256, 64)):
        with pytest.raises(G.RidgeGemmError):
            G.launch_form(*args)
    assert G.lib().ridge_gemm_launch_form(0, 256, 256, 64, 256, None) == G.HIP_ERROR_INVALID_VALUE


@pytest.mark.parametrize("absent", ["_cuda_getDevice", "_cuda_getCurrentRawStream"])
def test_the_current_stream_without_torchs_raw_calls(monkeypatch, absent):
    """A torch that lacks one of the raw calls: the public ones give the same handle."""
    torch = pytest.importorskip("torch")

    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream if device == 3 else None)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 3)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 77 if device == 3 else None)
    monkeypatch.delattr(torch._C, absent)
    monkeypatch.setattr(G, "_raw_calls", None, raising=False)
    assert G._stream_handle(None) == 77
