"""Where built libraries are looked for and written (no GPU)."""
import os
import re
import shutil
import stat
import subprocess

import pytest
import torch

from inferflux_amd.kernels import library


def test_the_fallback_folder_must_be_private_and_ours(tmp_path, monkeypatch):
    monkeypatch.setattr(library.tempfile, "gettempdir", lambda: str(tmp_path))
    d = tmp_path / f"inferflux_amd-{os.getuid()}"
    assert library._fallback_dir() is None and not d.exists()           # looking a library up creates nothing
    assert library._fallback_dir(create=True) == str(d) and stat.S_IMODE(os.lstat(d).st_mode) == 0o700
    os.chmod(d, 0o777)                                                   # others may write: whatever is in it is not trusted
    with pytest.raises(library.KernelBuildError, match="not a private folder"):
        library._fallback_dir()
    with pytest.raises(library.KernelBuildError, match="not a private folder"):
        library.find_library("ceilings", (("NO_SUCH_VARIANT", 1),))
    os.chmod(d, 0o700)
    os.rmdir(d)
    os.symlink(tmp_path, d)                                              # a link somebody planted under the expected name
    with pytest.raises(library.KernelBuildError, match="not a private folder"):
        library._fallback_dir(create=True)


def test_barriers_in_assembly_stand_behind_a_wait_for_what_was_read_from_lds():
    """A barrier written in assembly says that every wave is done reading a piece of LDS that is then overwritten.  Only the wait for the
    reads (lgkmcnt(0), in the same statement or as the builtin a few lines before) makes that so: the instructions that take what was read
    are no memory operations, so that the compiler may put them, and the waits it makes for them, behind the barrier."""
    found = 0
    for name in sorted(os.listdir(library.CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(library.CSRC, name)) as f:
            lines = f.read().split("\n")
        for i, line in enumerate(lines):
            if "asm" in line and "s_barrier" in line:
                found += 1
                before = "\n".join(lines[max(0, i - 5):i])
                assert "lgkmcnt(0)" in line.split("//")[0] or "__builtin_amdgcn_s_waitcnt(0xc07f)" in before, f"{name}:{i + 1}"
    assert found >= 4


def _sums_read_early(kernel, states=14):
    """Of a kernel's disassembled lines: those that may read an accumulation register fewer than ``states`` wait states (an instruction is one, s_nop n is n + 1)
    after a matrix product that writes it, on any path, branches taken and not."""
    def registers(operand):
        m = re.fullmatch(r"a(\d+)|a\[(\d+):(\d+)\]", operand)
        return set() if not m else {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))
    code, at = [], {}
    for line in kernel:
        text, _, comment = line.partition("//")
        op, _, rest = text.strip().partition(" ")
        target = re.search(r"<.*?(?:\+0x([0-9a-f]+))?>", comment) if op.startswith(("s_branch", "s_cbranch")) else None
        at[int(comment.split(":")[0], 16)] = len(code)
        code.append((op, [o.strip().split(" ")[0] for o in rest.split(",")], int(target[1] or "0", 16) if target else None, text.strip()))
    first = min(at)
    starts = {0} | {at[first + t] for _, _, t, _ in code if t is not None} | {i + 1 for i, c in enumerate(code) if c[2] is not None}
    since, todo, early = {0: {}}, [0], set()          # (where a block starts: registers written shortly before, with the states since)
    while todo:
        i = todo.pop()
        recent = dict(since[i])
        after = []
        while i < len(code):
            op, operands, target, text = code[i]
            if op.startswith("v_mfma"):
                recent = {**{r: n + 1 for r, n in recent.items() if n + 1 < states}, **dict.fromkeys(registers(operands[0]), 0)}
            else:
                read = set().union(*map(registers, operands if "store" in op or op.startswith("ds_write") else operands[1:]))
                if read & recent.keys():
                    early.add(text)
                took = int(operands[0], 0) + 1 if op == "s_nop" else 1
                recent = {r: n + took for r, n in recent.items() if n + took < states}
            i += 1
            if target is not None:
                after.append(at[first + target])
            if op in ("s_branch", "s_endpgm"):
                break
            if i in starts:
                after.append(i)
                break
        for j in after:
            known = since.get(j)
            joined = {r: min(n, (known or {}).get(r, states)) for r, n in recent.items()} | {r: n for r, n in (known or {}).items() if r not in recent}
            if joined != known:
                since[j] = joined
                todo.append(j)
    return early


def _line(address, text, target=None):
    return f"\t{text}  // {address:012X}: 00000000" + (f" <k+0x{target:x}>" if target is not None else "")


def test_sums_read_early_are_found_along_every_path():
    product, read = "v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[4:7]", "v_accvgpr_read_b32 v9, a6"
    assert _sums_read_early([_line(0, product), _line(8, read), _line(16, "s_endpgm")]) == {read}
    assert not _sums_read_early([_line(0, product), _line(8, "s_nop 12"), _line(12, read.replace("a6", "a8")), _line(16, read), _line(20, "s_endpgm")])
    assert _sums_read_early([_line(0, product), _line(8, "s_nop 12"), _line(12, read), _line(16, "s_endpgm")]) == {read}
    # around a loop, and over a branch to a place before
    assert _sums_read_early([_line(0, read), _line(8, "s_nop 15"), _line(16, product), _line(24, "s_cbranch_scc1 65530", 0), _line(32, "s_endpgm")]) == {read}
    assert _sums_read_early([_line(0, "s_branch 4", 24), _line(8, read), _line(16, "s_endpgm"), _line(24, product), _line(32, "s_cbranch_scc0 1", 8), _line(40, "s_nop 15"),
                             _line(48, read.replace("v9", "v8")), _line(56, "s_endpgm")]) == {read}
    assert _sums_read_early([_line(0, product), _line(8, "buffer_store_dwordx4 a[4:7], v1, s[0:3], 0 offen"), _line(16, "s_endpgm")])


@pytest.mark.parametrize("name", ["grouped_gemm", "gemm_tiles"])
def test_nothing_reads_a_sum_of_a_product_in_assembly_too_early(name, tmp_path):
    """The tiles by four large waves keep their sums in registers that products in assembly write.  The compiler does not know how long such a product takes,
    so a move of a sum that it puts shortly behind one (as it did with 256 items to a tile) reads what was there before: there is none in the built kernels."""
    dump, built = "/opt/rocm/llvm/bin/llvm-objdump", library.find_library(name)
    if built is None or not os.path.isfile(dump):
        pytest.skip("needs the built module and the disassembler")
    shutil.copy(built, tmp_path / "module.so")
    subprocess.run([dump, "--offloading", "module.so"], cwd=tmp_path, check=True, capture_output=True)
    image = next(f for f in os.listdir(tmp_path) if library.ARCH in f)
    text = subprocess.run([dump, "-d", "--no-show-raw-insn", image], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
    kernels = [k.split("\n") for k in re.split(r"\n(?=[0-9a-f]+ <)", text) if re.match(r"[0-9a-f]+ <.*(experts_waves|tiles)_kernel.*>:", k)]
    assert kernels
    for name_line, *lines in kernels:
        lines = [line for line in lines if "//" in line]
        assert sum("v_mfma" in line for line in lines) > 50
        assert not _sums_read_early(lines), name_line


class _Function:
    """A function of ``types`` (p, a, i, l, f) in a module of its own that keeps what it is called with and returns ``rc``."""

    def __init__(self, types, rc=0):
        import ctypes

        from inferflux_amd.kernels import ops
        words = {"p": ops.P, "a": ops.P, "i": ops.I, "l": ops.LL, "f": ops.F}
        self.got, self.name, self.entries = None, "fake", {}
        self.argtypes = tuple(ctypes.POINTER(ops.I) if c == "a" else words[c] for c in types)

        def record(*args):
            self.got = args
            return rc
        self.keep = ctypes.CFUNCTYPE(ctypes.c_int, *(words[c] for c in types))(record)

    def fn(self, fname, argtypes):
        return self.keep

    def last_error(self):
        return "an error of its own"


@pytest.mark.parametrize("types", ["", "p", "f", "pppppp", "ppppppp", "ffffffff", "pifpifpifl", "iiiiiiiiiifffffffflp",
                                   "pppppppppppiiiiiiiifiippppiiiippiif", "i" * 38, "l" * 38 + "f" * 8])
def test_native_calls_pass_what_ctypes_passes(types):
    import ctypes
    import random
    import struct

    from inferflux_amd.kernels import ops
    rng, t = random.Random(len(types)), torch.arange(6, dtype=torch.int32)
    f = _Function(types)
    args, want = [], []
    for c in types:
        if c == "p":
            v = rng.choice([None, 0, t, 0x7fff12345678, (1 << 64) - 16])
            args.append(v)
            want.append((v.data_ptr() if v is t else v) or None)
        elif c == "f":
            args.append(rng.choice([1, 0.1, -3.5e30, float("inf"), 2 ** -149]))
            want.append(struct.unpack("f", struct.pack("f", float(args[-1])))[0])
        else:
            args.append(rng.choice([0, -1, True, 2 ** 31 - 1, -2 ** 31] + ([2 ** 40 + 3] if c == "l" else [])))
            want.append(int(args[-1]))
    ops._call(f, "fake", f.argtypes, *args)
    assert "fake" in f.entries and f.entries["fake"] is not None
    assert list(f.got) == want
    f.got = None
    ops._call(f, "fake", f.argtypes, *args)              # (by what was kept of the first call)
    assert list(f.got) == want
    assert ctypes.sizeof(ctypes.c_void_p) == 8


def test_native_calls_leave_the_rest_to_ctypes():
    import ctypes

    import numpy as np

    from inferflux_amd.kernels import ops
    f = _Function("iaf")
    ints = (ctypes.c_int * 3)(4, 5, 6)
    ops._call(f, "fake", f.argtypes, 1, ints, 2.0)       # (the address of an array)
    assert f.got[1] == ctypes.addressof(ints) and f.got[0::2] == (1, 2.0)
    f = _Function("i" * 39)                              # more than the native call has places for
    ops._call(f, "fake", f.argtypes, *range(39))
    assert f.entries["fake"] is None and f.got == tuple(range(39))
    for wrong in ((1,), ("one", 2.0), (1, "two"), (np.int64(1), None)):
        g = _Function("if")
        g.keep.argtypes = list(g.argtypes)
        with pytest.raises((TypeError, ctypes.ArgumentError)):
            ops._call(g, "fake", g.argtypes, *wrong)
        assert g.got is None
    g = _Function("if")
    g.keep.argtypes = list(g.argtypes)
    with pytest.raises((TypeError, ctypes.ArgumentError)):                   # (what comes after is converted by ctypes' own rules, too)
        ops._call(g, "fake", g.argtypes, 1, 2.0, "three", object())
    g = _Function("if")
    ops._call(g, "fake", g.argtypes, 1, 2.0, 3)          # (a C function called with more than it takes, which ctypes allows)
    assert g.got[:2] == (1, 2.0)
    f = _Function("p", rc=-7)
    with pytest.raises(ops.KernelError, match=r"fake: an error of its own \(code -7\)"):
        ops._call(f, "fake", f.argtypes, None)


def test_native_calls_take_a_pointers_array_only_as_ctypes_does():
    """For a pointer to 32-bit numbers: an array of them by its address, a pointer by what it points to (an object's own buffer would be the pointer
    itself), None as none, and nothing else."""
    import ctypes

    import numpy as np

    from inferflux_amd.kernels import ops

    def given(v):
        f = _Function("ia")
        f.keep.argtypes = list(f.argtypes)
        got = []
        f.keep = ctypes.CFUNCTYPE(ctypes.c_int, ops.I, ctypes.POINTER(ops.I))(lambda i, p: got.append(ctypes.cast(p, ops.P).value) or 0)
        ops._call(f, "fake", f.argtypes, 1, v)
        return got[0]
    ints = (ctypes.c_int * 3)(4, 5, 6)
    numbers = np.arange(3, dtype=np.int32)
    assert given(ints) == ctypes.addressof(ints) and given(None) is None
    first = ctypes.c_int.from_buffer(ints)
    for pointer in (ctypes.cast(ints, ctypes.POINTER(ctypes.c_int)), ctypes.pointer(first), ctypes.byref(first)):
        assert given(pointer) == ctypes.addressof(ints)
    assert given(numbers.ctypes.data_as(ctypes.POINTER(ctypes.c_int))) == numbers.ctypes.data
    for wrong in (numbers, np.arange(3), b"ab", bytearray(8), (ctypes.c_float * 3)(), (ctypes.c_longlong * 2)(), memoryview(b"abcd")):
        with pytest.raises(ctypes.ArgumentError):
            given(wrong)


def test_native_checks_raise_what_the_python_check_raises():
    from inferflux_amd.kernels import ops
    x = torch.zeros(2, 3)
    for args in ((3, "x"), (x, "x"), (x, "x", (2, 3)), (x, "x", None, torch.float32), (x.t(), "x", (3, 2), torch.float64), (None, "x", (None,))):
        with pytest.raises(ops.KernelError) as a:
            ops._check_in_python(*args)
        with pytest.raises(ops.KernelError) as b:
            ops._check(*args)
        assert str(a.value) == str(b.value)
    with pytest.raises(ops.KernelError):
        ops._check(x, "x", dtype=torch.float32)          # (keywords, too)
    y = ops.empty((2, 0, 5), torch.bfloat16, x)
    assert y.shape == (2, 0, 5) and y.dtype == torch.bfloat16 and y.device == x.device and y.is_contiguous()
    for wrong in (((2,), torch.int32), ([2], torch.int32, x), ((2,), "int32", x), ((2,), torch.int32, None), ((2.5,), torch.int32, x), ((-1,), torch.int32, x)):
        with pytest.raises((TypeError, RuntimeError)):
            ops.empty(*wrong)


@pytest.mark.parametrize("failure", [library.KernelBuildError("g++ failed\nwith many lines"), ImportError("built for another interpreter"), OSError("no such library")])
def test_without_the_native_calls_python_does_their_work(failure, capfd):
    """A host that cannot build the extension imports the package all the same: the same checks, calls and tensors by the Python forms, and a line that says so."""
    from inferflux_amd.kernels import ops

    def load(name):
        raise failure
    native, check, call, empty, stream = ops._host_forms(load)
    assert native is None and str(failure).split("\n")[0] in capfd.readouterr().err
    x = torch.zeros(2, 3)
    with pytest.raises(ops.KernelError, match="GPU"):
        check(x, "x", (2, 3))
    y = empty((2, 0, 5), torch.bfloat16, x)
    assert y.shape == (2, 0, 5) and y.dtype == torch.bfloat16 and y.device == x.device
    f = _Function("pif")
    call(f, "fake", f.argtypes, x, 7, 0.5)
    assert f.got == (x.data_ptr(), 7, 0.5) and callable(stream)
    f = _Function("p", rc=-7)
    with pytest.raises(ops.KernelError, match=r"fake: an error of its own \(code -7\)"):
        call(f, "fake", f.argtypes, None)


def test_the_package_imports_where_nothing_can_be_built(tmp_path):
    """Its configurations and plans do not need a compiler: a copy of the Python files alone, with no compiler to be found."""
    import sys
    root = os.path.dirname(os.path.dirname(library.CSRC))
    shutil.copytree(os.path.join(root, "inferflux_amd"), tmp_path / "inferflux_amd", ignore=shutil.ignore_patterns("*.so", "__pycache__", ".*.lock"))
    env = {**os.environ, "PATH": "", "CXX": "/nonexistent", "HIPCC": "", "ROCM_PATH": "/nonexistent", "TMPDIR": str(tmp_path), "PYTHONDONTWRITEBYTECODE": "1"}
    code = ("from inferflux_amd.kernels import library\n"
            "def absent():\n    raise library.KernelBuildError('no compiler')\n"
            "library._cxx = absent\n"
            "from inferflux_amd.engine import engine, context\n"
            "from inferflux_amd.kernels import ops\n"
            "print('native', ops._native)\n")
    out = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env=env, capture_output=True, text=True, timeout=110)
    assert out.returncode == 0 and "native None" in out.stdout and "no compiler" in out.stderr, out.stderr[-2000:]


@pytest.mark.gpu
def test_native_checks_on_the_gpu():
    from inferflux_amd.kernels import ops
    x = torch.zeros(4, 6, device="cuda")
    tensors = (x, x.t(), x[:, :3], x[1:3], x.bfloat16(), x[0], x[0, 0], torch.empty(0, 6, device="cuda"), torch.nn.Parameter(x))
    shapes = (None, (4, 6), (None, 6), (4, None), (None, None), (6,), (), (2, 6), [4, 6], (4, 6, 1), x.shape, (0, None))
    for t in tensors:
        for shape in shapes:
            for dtype in (None, torch.float32, torch.bfloat16):
                def outcome(f):
                    try:
                        f(t, "t", shape, dtype)
                    except ops.KernelError as e:
                        return str(e)
                assert outcome(ops._check) == outcome(ops._check_in_python), (t.shape, shape, dtype)
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert ops._stream() == side.cuda_stream != 0
    a = ops.upload(__import__("numpy").arange(1000, dtype="int32"), x.device)
    assert torch.equal(a.cpu(), torch.arange(1000, dtype=torch.int32))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):                  # (from ordinary memory the copy was refused there, too)
        b = a + 1
        with pytest.raises(ops.KernelError, match="captured"):
            ops.upload(__import__("numpy").arange(1000, dtype="int32"), x.device)
    for n in (1, 2):
        a += 1
        graph.replay()
        assert torch.equal(b.cpu(), torch.arange(1000, dtype=torch.int32) + n + 1)
