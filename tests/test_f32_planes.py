"""kernels/matmul_f32_split.hip, the fp32 products of a plan on the bf16 matrix pipes: ragged and whole rows,
columns and depths (its end 1, 31 and 32 deep), every layout, 64x64 and 128x128 tiles, a depth dealt to
workgroups.  Against the product in float64, element by element, within the rounding of K fp32
additions and products (K * 2^-24 * sum of |a b|); no further off than the fp32 MFMA; infinities, NaN and values too
small for three bf16 planes to hold as the fp32 MFMA has them."""
import ctypes as C
import os
import re
import subprocess
import sys
import tempfile

import pytest

import hostcheck
from polygrad_amd import PlanFile, _ffi

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "perf"))
import cases  # noqa: E402

PLAN = 8      # poly_hip_render and poly_hip_describe: as a kernel of a plan
SHAPES = [(1025, 1024, 64, "nt", "64x64"), (1030, 1040, 97, "nn", "64x64"), (1088, 992, 127, "tn", "64x64"), (1056, 1000, 65, "tt", "64x64"),
          (1793, 1664, 129, "nn", "128x128"), (1801, 1700, 160, "tn", "128x128"), (1665, 1793, 191, "nt", "128x128"), (1700, 1799, 128, "tt", "128x128"),
          (1024, 1024, 2048, "nn", "128x128"), (1008, 1008, 3072, "tn", "128x128"), (512, 3070, 768, "nt", "128x128")]


def _case(c):
    return dict(kind="matmul", m=c[0], n=c[1], k=c[2], dtype="float32", layout=c[3])


def _is_it(desc, c):
    dealt = re.search(r"K dealt to (\d+)", desc)
    return "three planes of each f32 value" in desc and f"tile {c[4]}x32" in desc and (dealt is not None) == (c[2] >= 768)


def check_as_of_a_plan(hiplib, schedule, item, pieces=None):
    """The kernel of `item` as a plan has it, and its first stages, on the host with buffers of their exact size, or
    of some of them only the pieces that there are (hostcheck.check_kernel)."""
    launch = (C.c_int * 7)()
    units = _ffi.take_string(hiplib.poly_hip_render(item.root, b"k", PLAN, launch)).split("\n// ---- ")
    sizes, scratch = [schedule.buf_slots[item.buf_slot_indices[p]].nbytes for p in range(item.n_buf_slots)], 0
    jobs = [(units[0], (launch[0], launch[1], launch[2]), launch[3])]
    for u in units[1:]:
        m = re.match(r"first stage ---- grid=(\d+),(\d+) block=(\d+) scratch=(\d+)\n", u)
        scratch = int(m.group(4))
        jobs.append((u[m.end():], (int(m.group(1)), int(m.group(2)), 1), int(m.group(3))))
    for source, grid, block in jobs:
        hostcheck.check_kernel(source, hostcheck._entry_name(source), grid, block, sizes, block_stride=max(1, grid[0] * grid[1] * block // (1 << 17)), scratch_bytes=scratch, pieces=pieces)


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_stays_in_bounds(c, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    pf = cases._matmul_schedule(_case(c)).plan()
    s = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents
    it = s.items[0]
    assert _is_it(_ffi.take_string(hiplib.poly_hip_describe(it.root, PLAN)), c)
    assert "three planes" not in _ffi.take_string(hiplib.poly_hip_describe(it.root, 0))
    check_as_of_a_plan(hiplib, s, it)


def _scratch_bytes(source):
    """Of scratch memory to a lane, in the code object that the run-time compiler makes of `source`."""
    rtc, prog, size = C.CDLL("/opt/rocm/lib/libhiprtc.so"), C.c_void_p(), C.c_size_t()
    options = (C.c_char_p * 8)(*b"--offload-arch=gfx950 -O3 -std=c++17 -ffp-contract=off -Xclang -target-feature -Xclang -packed-fp32-ops".split())
    assert rtc.hiprtcCreateProgram(C.byref(prog), source.encode(), b"k.hip", 0, None, None) == 0
    assert rtc.hiprtcCompileProgram(prog, 8, options) == 0
    rtc.hiprtcGetCodeSize(prog, C.byref(size))
    code = C.create_string_buffer(size.value)
    rtc.hiprtcGetCode(prog, code)
    rtc.hiprtcDestroyProgram(C.byref(prog))
    with tempfile.NamedTemporaryFile() as f:
        f.write(code.raw)
        f.flush()
        notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", f.name], capture_output=True, text=True, check=True).stdout
    return int(re.search(r"\.private_segment_fixed_size: +(\d+)", notes).group(1))


@pytest.mark.skipif(not os.path.exists("/opt/rocm/llvm/bin/llvm-readelf"), reason="no reader of code objects")
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,ks", [(320, 3776, (74, 82, 90, 372)), (1793, 1664, (129, 138, 148, 157))])
def test_ends_of_the_depth_stay_in_registers(m, n, ks, layout, hiplib, monkeypatch):
    monkeypatch.setattr(cases, "HipPlan", type("Loader", (), {"from_file": staticmethod(PlanFile)}))
    for k in ks:
        pf = cases._matmul_schedule(dict(kind="matmul", m=m, n=n, k=k, dtype="float32", layout=layout)).plan()
        it = C.cast(pf.schedule, C.POINTER(_ffi.PolySchedule)).contents.items[0]
        if "three planes" in _ffi.take_string(hiplib.poly_hip_describe(it.root, PLAN)):      # (rows of an odd number of lines are another template's)
            assert _scratch_bytes(_ffi.take_string(hiplib.poly_hip_render(it.root, b"k", PLAN, None)).split("\n// ---- ")[0]) == 0


def _product(c, change=None):
    state = cases.prepare(_case(c), 9)
    by = {s.name: state["data"][s.index] for s in state["plan"].external_slots()}
    if change:
        change(by["A"], by["B"])
    got = cases.run(state)["C"]
    state["plan"].sync()
    m, n, k, layout = c[:4]
    a = by["A"].reshape(k, m).T if layout[0] == "t" else by["A"].reshape(m, k)
    b = by["B"].reshape(n, k).T if layout[1] == "t" else by["B"].reshape(k, n)
    return state["plan"].kernel_info()[0]["desc"], got.reshape(m, n).cpu(), a.double().cpu(), b.double().cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_against_float64(c, monkeypatch):
    desc, got, a, b = _product(c)
    assert _is_it(desc, c)
    want = a @ b
    err = (got.double() - want).abs()
    assert bool((err <= c[2] * 2.0 ** -24 * (a.abs() @ b.abs())).all())
    monkeypatch.setenv("POLY_HIP_NO_F32_SPLIT", "1")
    desc, there, _, _ = _product(c)
    assert "three planes" not in desc
    assert float(err.norm()) <= float((there.double() - want).norm())


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["inf", "nan", "largest", "tiny", "overflow"])
@pytest.mark.parametrize("c", [SHAPES[1], SHAPES[4], SHAPES[8]], ids=lambda c: "-".join(map(str, c)))
def test_values_that_planes_do_not_hold(c, what, monkeypatch):
    """The same infinities and NaN as the fp32 MFMA, and finite values within the rounding of both."""
    import torch

    def change(a, b):
        if what == "inf":
            a[5], a[4000], b[77] = float("inf"), -float("inf"), float("inf")
        elif what == "nan":
            a[5], b[77] = float("nan"), float("nan")
        elif what == "largest":
            a[5] = torch.finfo(torch.float32).max
            b.mul_(2.0 ** -30)
        elif what == "tiny":
            a.mul_(2.0 ** -118)
        else:
            a[5] = 3e38
            b[77] = 3e38
    desc, got, a, b = _product(c, change)
    assert _is_it(desc, c)
    monkeypatch.setenv("POLY_HIP_NO_F32_SPLIT", "1")
    _, want, _, _ = _product(c, change)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    finite = want.isfinite()
    assert torch.equal(got[~finite & ~want.isnan()], want[~finite & ~want.isnan()])
    a, b = a.nan_to_num(0.0, 0.0, 0.0), b.nan_to_num(0.0, 0.0, 0.0)
    # (below the smallest normal number a product's rounding is absolute)
    bound = 2 * c[2] * (2.0 ** -24 * (a.abs() @ b.abs()) + 2.0 ** -149)
    assert bool(((got.double() - want.double()).abs() <= bound)[finite].all())


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["whole", "smallest"])
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_rows_of_one_term(c, what):
    """One rounding of the one product of each sum: of the nine products of planes eight are there (the ninth is 2^-34
    of it), and the sums of the seven behind the leading one, 2^-7 of it at most, are rounded seven times.  Also of the smallest
    values that planes hold, 2^-110 to 2^-104, the last plane of which is below the smallest normal number."""
    import torch
    m, n, k = c[:3]

    def change(a, b):
        a2 = a.view(k, m).T if c[3][0] == "t" else a.view(m, k)
        at = (torch.arange(m, device="cuda"), torch.randint(0, k, (m,), device="cuda"))
        one = a2[at].sign() * (a2[at].abs().fmod(1.0) + 1.0)
        if what == "smallest":
            one *= 2.0 ** torch.randint(-110, -104, (m,), device="cuda").double()
            b.mul_(2.0 ** 60)
        a2.zero_()
        a2[at] = one
    desc, got, a, b = _product(c, change)
    assert _is_it(desc, c)
    want = a @ b
    assert bool(((got.double() - want).abs() <= 2.0 ** -24 * (1 + 2.0 ** -4) * want.abs()).all())


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [2.0 ** -108, 2.0 ** -66])
@pytest.mark.parametrize("c", [SHAPES[1], SHAPES[4], SHAPES[8]], ids=lambda c: "-".join(map(str, c)))
def test_small_values_beside_ones_that_planes_do_not_hold(c, scale):
    """Values about the smallest that planes hold, times large ones, one of them below it, and values whose products are
    about the smallest normal number: within the rounding of K additions and products, of a product below that number
    an absolute one."""
    def change(a, b):
        a.mul_(scale)
        a[4000] = 2.0 ** -111
        b.mul_(2.0 ** 60 if scale < 2.0 ** -100 else scale)
    desc, got, a, b = _product(c, change)
    assert _is_it(desc, c)
    err = (got.double() - a @ b).abs()
    assert bool((err <= c[2] * (2.0 ** -24 * (a.abs() @ b.abs()) + 2.0 ** -149)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("c", SHAPES, ids=lambda c: "-".join(map(str, c)))
def test_tiles_that_are_computed_again_against_float64(c, monkeypatch):
    """A value below 2^-110 in every row sends every tile to the fp32 MFMA: within the rounding of K additions and
    products, and no further off than the fp32 templates are (whose sums are as many, of other terms: a twentieth for
    that)."""
    def change(a, b):
        (a.view(c[2], c[0])[c[2] // 2] if c[3][0] == "t" else a.view(c[0], c[2])[:, c[2] // 2]).fill_(2.0 ** -112)
    desc, got, a, b = _product(c, change)
    assert _is_it(desc, c)
    want = a @ b
    err = (got.double() - want).abs()
    assert bool((err <= c[2] * 2.0 ** -24 * (a.abs() @ b.abs())).all())
    monkeypatch.setenv("POLY_HIP_NO_F32_SPLIT", "1")
    desc, there, _, _ = _product(c, change)
    assert "three planes" not in desc
    assert float(err.norm()) <= 1.05 * float((there.double() - want).norm())
