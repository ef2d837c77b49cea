"""The kernels on the CPU (no GPU): host_exec/ builds the library against a
small stand-in for the HIP runtime and runs every block of every launch under
the address sanitizer, in three thread orders. An access out of range, a value
used before it is written, a missing barrier and a written layout gap all fail
here; the values are compared with FP64 references."""
import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import scipy.fft as sf

from gpu_util import TOL, bf16_bits, bf16_to_f32, span
from plfft_amd import rng as prng

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "perf-libs-fft_amd", "csrc")
HOST = os.path.join(ROOT, "tests", "host_exec")
CXX = "/opt/rocm/llvm/bin/clang++"
FLAGS = ["-std=c++17", "-O0", "-g1", "-Xarch_host", "-fsanitize=address",
         "-ftrivial-auto-var-init=pattern", "-w", "-I", HOST, "-I", os.path.join(ROOT, "include")]
STORE = {"f32": np.float32, "f64": np.float64, "f16": np.float16, "bf16": np.uint16}
R2R = {"dct2": 1, "dct3": 2, "dst2": 5, "dst3": 6}
pytestmark = pytest.mark.skipif(not os.path.exists(CXX), reason="no ROCm clang")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_exec")

    def compile_one(src):
        obj = str(d / (os.path.basename(src) + ".o"))
        subprocess.run([CXX, "-x", "c++", *FLAGS, "-c", src, "-o", obj], check=True)
        return obj

    src = [os.path.join(CSRC, f) for f in sorted(os.listdir(CSRC)) if f.endswith((".hip", ".cpp"))]
    with ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
        objs = list(pool.map(compile_one, src + [os.path.join(HOST, "host_exec.cpp")]))
    out = str(d / "host_exec")
    subprocess.run([CXX, *FLAGS, "-o", out, *objs], check=True)
    yield out
    shutil.rmtree(d, ignore_errors=True)


def _store(x, dtype):
    return bf16_bits(x.astype(np.float32)) if dtype == "bf16" else x.astype(STORE[dtype])


def _value(b, dtype):
    return (bf16_to_f32(b) if dtype == "bf16" else b).astype(np.float64)


class Side:
    """One side of a plan: count elements at stride, howmany members at dist."""

    def __init__(self, count, stride, howmany, dist, real):
        w = 1 if real else 2
        self.real, self.size = real, w * span(count, stride, howmany, dist)
        e = np.arange(howmany)[:, None] * dist + np.arange(count)[None, :] * stride
        self.at = w * e
        self.used = np.zeros(self.size, bool)
        for i in range(w):
            self.used[self.at + i] = True

    def members(self, flat):
        return flat[self.at] if self.real else flat[self.at] + 1j * flat[self.at + 1]


def _forward(kind, n, direction, r2r, x):
    if kind == "c2c":
        return np.fft.fft(x) if direction < 0 else np.fft.ifft(x, norm="forward")
    if kind == "r2c":
        return np.fft.rfft(x)
    if kind == "c2r":
        return np.fft.irfft(x, n=n, norm="forward")
    return (sf.dct if r2r[:3] == "dct" else sf.dst)(x, int(r2r[3]))


def _adjoint(kind, n, direction, r2r, g):
    """Transpose of the real-linear map (C2C: conjugate transpose)."""
    if kind == "c2c":
        return _forward("c2c", n, -direction, r2r, g)
    if kind == "r2c":
        full = np.zeros((len(g), n), complex)
        full[:, :n // 2 + 1] = g
        return np.fft.ifft(full, norm="forward").real
    if kind == "c2r":
        y = 2.0 * np.fft.rfft(g)
        ends = [0, -1] if n % 2 == 0 else [0]
        y[:, ends] = 0.5 * y[:, ends].real
        return y
    return g @ _forward(kind, n, direction, r2r, np.eye(n)).T


def P(kind, n, howmany, dtype="f32", direction=-1, lay=None, adjoint=0, inplace=0, cus=256,
      node=""):
    """lay: (istride, idist, ostride, odist), "cols", or None (packed)."""
    r2r = kind if kind in R2R else ""
    kind = "r2r" if r2r else kind
    ic, oc = (n // 2 + 1 if kind == "c2r" else n), (n // 2 + 1 if kind == "r2c" else n)
    if lay is None:
        lay = (1, ic, 1, oc)
    elif lay == "cols":
        lay = (howmany, 1, howmany, 1)
    return dict(kind=kind, n=n, howmany=howmany, dtype=dtype, direction=direction, r2r=r2r,
                lay=lay, ic=ic, oc=oc, adjoint=adjoint, inplace=inplace, cus=cus, node=node)


def run(exe, tmp_path, cases):
    lines, todo = [], []
    for i, c in enumerate(cases):
        rng = np.random.default_rng(i)
        fin, fout = str(tmp_path / f"c{i}.in"), str(tmp_path / f"c{i}.out")
        dt = c["dtype"]
        size = np.dtype(STORE[dt]).itemsize
        lines.append(f"cus {c.get('cus', 256)}")
        if "lengths" in c:
            total = 2 * sum(c["lengths"])
            x = _store(rng.standard_normal(total), dt)
            lines.append(f"mixed c{i} {len(c['lengths'])} {dt} {c['direction']} {c['inplace']} " +
                         " ".join(map(str, c["lengths"])) + f" {total * size} {fin} {fout}")
        else:
            (si, di, so, do), hm = c["lay"], c["howmany"]
            src = Side(c["ic"], si, hm, di, c["kind"] in ("r2c", "r2r"))
            dst = Side(c["oc"], so, hm, do, c["kind"] in ("c2r", "r2r"))
            if c["adjoint"]:
                src, dst = dst, src
            c["src"], c["dst"] = src, dst
            x = _store(rng.standard_normal(src.size), dt)
            lines.append(f"plan c{i} {c['kind']} {c['n']} {hm} {dt} {c['direction']} "
                         f"{R2R.get(c['r2r'], 0)} {si} {di} {so} {do} {c['adjoint']} "
                         f"{c['inplace']} {dst.size * size} {fin} {fout}")
        x.tofile(fin)
        todo.append((c, x, fout))
    r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-300:] + r.stderr[-4000:]
    plans = dict(line.split(" ", 1) for line in r.stdout.splitlines() if line[0] == "c")
    for i, (c, x, fout) in enumerate(todo):
        dt = c["dtype"]
        y = np.fromfile(fout, STORE[dt])
        xv, yv = _value(x, dt), _value(y, dt)
        if "lengths" in c:
            o = 0
            for n in c["lengths"]:
                m = slice(2 * o, 2 * (o + n))
                ref = _forward("c2c", n, c["direction"], "", xv[m].view(np.complex128))
                _close(yv[m].view(np.complex128), ref, TOL[dt], (n, plans[f"c{i}"]))
                o += n
            continue
        assert c["node"] in plans[f"c{i}"], plans[f"c{i}"]
        f = _adjoint if c["adjoint"] else _forward
        ref = f(c["kind"], c["n"], c["direction"], c["r2r"], c["src"].members(xv))
        _close(c["dst"].members(yv), ref, TOL[dt], plans[f"c{i}"])
        size = y.dtype.itemsize
        before = np.full(len(y) * size, 0xA5, np.uint8)
        if c["inplace"]:
            k = min(x.nbytes, len(before))
            before[:k] = x.view(np.uint8)[:k]
        gap = ~c["dst"].used
        assert np.array_equal(y.view(np.uint8).reshape(-1, size)[gap],
                              before.reshape(-1, size)[gap]), plans[f"c{i}"]


def _close(y, ref, tol, what):
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert err <= tol, (err, what)  # a NaN fails too


@pytest.mark.parametrize("which,word", [(0, None), (1, "use-after-poison"), (2, "order of the threads"),
                                        (3, "barrier"), (4, "heap-buffer-overflow")])
def test_planted_faults_are_found(exe, tmp_path, which, word):
    r = subprocess.run([exe], input=f"fault {which} {tmp_path / 'y'}\n", capture_output=True, text=True)
    assert (r.returncode == 0) == (word is None), r.stderr[-2000:]
    assert word is None or word in r.stderr, r.stderr[-2000:]


ALL = ["f32", "f64", "f16", "bf16"]
REAL_PAD = {"r2c": lambda n: (1, 2 * (n // 2 + 1), 1, n // 2 + 1),
            "c2r": lambda n: (1, n // 2 + 1, 1, 2 * (n // 2 + 1))}  # in place


@pytest.mark.parametrize("dtype", ALL)
def test_columns_and_four_step(exe, tmp_path, dtype):
    wide = {"f32": 16, "f64": 8, "f16": 16, "bf16": 16}[dtype]
    run(exe, tmp_path, [
        # tile kernels (few CUs, so that a short batch takes them): last tile partial, row pitch
        # of any length (tiles in XCD order), in place
        P("c2c", 64, 300, dtype, -1, "cols", cus=8, node="tile_c2c"),
        P("c2c", 256, 65, dtype, 1, "cols", cus=8, node="tile_c2c", inplace=1),
        P("c2c", 1024, 3 * wide + 1, dtype, -1, (3 * wide + 6, 1, 3 * wide + 3, 1), cus=8,
          node="tile_c2c"),
        P("c2c", 65536, 2, dtype, -1, (1, 65539, 1, 65536), cus=8, node="tile_col"),
        P("c2c", 65536, 1, dtype, 1, cus=8, node="tile_col", inplace=1),
    ])


@pytest.mark.parametrize("dtype", ALL)
def test_flexible_chains(exe, tmp_path, dtype):
    cases = [P("c2c", n, hm, dtype, d, inplace=k)
             for n, hm, d, k in ((2, 5, -1, 0), (13, 70, 1, 1), (60, 49, -1, 1), (100, 7, 1, 0),
                                 (1000, 6, -1, 1), (3000, 2, 1, 1), (1001, 3, -1, 0))]
    cases += [P("c2c", 100, 149, dtype, -1, "cols", node="lanes"),
              P("c2c", 60, 33, dtype, 1, (35, 1, 33, 1), node="lanes"),
              P("c2c", 1000, 17, dtype, 1, "cols", inplace=1, node="lanes"),
              # two and three members a block
              P("c2c", {"f64": 2000}.get(dtype, 3000), 65, dtype, -1, "cols", node="lanes"),
              P("c2c", 360, 9, dtype, -1, (2, 725, 3, 1081))]
    run(exe, tmp_path, cases)


@pytest.mark.parametrize("dtype", ALL)
def test_real_transforms(exe, tmp_path, dtype):
    cases = []
    for n, hm in ((4, 9), (60, 21), (100, 8), (1000, 5), (6000, 2), (33, 4)):
        for kind in ("r2c", "c2r"):
            cases += [P(kind, n, hm, dtype, lay=REAL_PAD[kind](n), inplace=1),
                      P(kind, n, hm, dtype, adjoint=1)]
    for n, hm in ((16, 700), (64, 70), (128, 33), (4096, 3)):
        cases += [P("r2c", n, hm, dtype), P("c2r", n, hm, dtype)]
    # (one CU: the line above which short members pass through LDS)
    cases += [P(k, n, hm, dtype, cus=1) for n, hm in ((64, 1030), (128, 517)) for k in ("r2c", "c2r")]
    cases += [P("r2c", 512, hm, dtype, lay=(2, 1025, 1, 257)) for hm in (1, 17)]
    cases += [P("c2r", 512, hm, dtype, lay=(2, 515, 1, 512)) for hm in (1, 17)]
    cases += [P("r2c", 100, 5, dtype, lay=(2, 211, 1, 53)), P("c2r", 100, 5, dtype, lay=(1, 53, 3, 301))]
    run(exe, tmp_path, cases)


@pytest.mark.parametrize("dtype", ALL)
def test_cosine_and_sine_transforms(exe, tmp_path, dtype):
    run(exe, tmp_path, [P(kind, n, hm, dtype, lay=lay, adjoint=adj, inplace=k)
                        for kind in R2R
                        for n, hm, lay, adj, k in ((200, 5, None, 0, 0), (200, 5, (2, 464, 1, 200), 1, 0),
                                                   (1000, 3, None, 1, 0), (60, 9, None, 0, 1),
                                                   (256, 9, (2, 576, 1, 256), 1, 0), (45, 6, None, 0, 0))])


@pytest.mark.parametrize("dtype", ALL)
def test_convolutions(exe, tmp_path, dtype):
    # one block (Rader, Bluestein), three passes (Rader 12289, chirp-z 10007 and
    # 20011: rows of 96, 192 and 384 in FP64)
    run(exe, tmp_path, [P("c2c", n, hm, dtype, d, inplace=k)
                        for n, hm, d, k in ((17, 300, -1, 0), (97, 17, 1, 1), (59, 33, -1, 0),
                                            (509, 3, 1, 0), (1009, 2, -1, 1), (1399, 2, 1, 0),
                                            (12289, 1, -1, 1), (10007, 2, 1, 0),
                                            (20011, 1, -1, 0))] + (
        # Bluestein of few members (8 points a thread) and of many (16)
        [P("c2c", n, hm, dtype, -1, node=f"bluestein_f64_fwd_n{M}_r{r}_t", cus=c)
         for n, M, hm, c, r in ((58, 128, 9, 256, "8x2x8"), (58, 128, 40, 2, "16x8"),
                                (458, 1024, 3, 256, "8x2x8x8"), (458, 1024, 9, 2, "16x4x16"),
                                (838, 2048, 3, 256, "8x4x8x8"), (838, 2048, 5, 2, "16x8x16"))]
        if dtype == "f64" else []))


@pytest.mark.parametrize("dtype,direction,inplace", [("f32", -1, 0), ("f32", 1, 1), ("f64", -1, 0),
                                                     ("f16", 1, 0), ("bf16", -1, 1)])
def test_mixed_batches(exe, tmp_path, dtype, direction, inplace):
    lengths = prng.mixed_lengths(7, 24, hi=20000) + [1, 2, 4096, 8192, 10007, 3 * 1009, 2 * 1999]
    run(exe, tmp_path, [dict(lengths=lengths, dtype=dtype, direction=direction, inplace=inplace,
                             cus=c) for c in (256, 2)])


def describe(exe, kind, n, howmany, dtype, lay):
    line = f"plan c {kind} {n} {howmany} {dtype} -1 0 {' '.join(map(str, lay))} 0 0 0 - -\n"
    r = subprocess.run([exe], input=line, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.split(" ", 1)[1]


# kind, length, output distance, what bounds the input side (elements of one or two reals), types
LIMITED = [(k, n, od, w, dt) for k, n, od, w, types in
           (("c2c", 1000, 1000, 2, ("f32", "f64", "f16")), ("r2c", 1000, 501, 1, ("f32", "f64")),
            ("c2r", 1000, 1000, 2, ("f32", "f64")), ("c2c", 256, 256, 2, ("f32", "f16")),
            ("c2c", 1024, 1024, 2, ("f32", "f16")))
           for dt in types]


@pytest.mark.parametrize("kind,n,od,w,dtype", LIMITED)
def test_distances_beyond_32_bit_offsets(exe, kind, n, od, w, dtype):
    """A block's members are addressed with 32-bit byte offsets: from the first
    distance on whose block reaches 2^32 bytes another kernel is chosen."""
    def name(idist, odist):
        return describe(exe, kind, n, 100000, dtype, (1, idist, 1, odist)).split()[0]

    near = name(2 * n, od)
    assert "flex" in near or "unit" in near
    tpb = int(near.split("_b")[1].split("_")[0])
    assert tpb > 1
    # the distance at which the block's end lies at 2^32 bytes
    last = 2 ** 32 // (w * np.dtype(STORE[dtype]).itemsize * tpb)
    assert name(last - 2 * n, od) == near and name(last, od) != near
    if kind == "c2c":
        assert name(2 * n, last - 2 * n) == near and name(2 * n, last) != near
