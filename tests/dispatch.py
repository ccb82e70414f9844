"""Which kernels a call launches, seen without a GPU: `launched` runs entry
points in a process of their own over a recording stand-in for the HIP runtime
(hip_stub.c), with addresses that nothing reads."""
import ctypes
import json
import os
import re
import subprocess
import sys
import tempfile
import types

HERE = os.path.dirname(os.path.abspath(__file__))
ADDR = 0x10000000  # any 16-byte aligned address


def launched(steps, want="launches"):
    """Per step, the launches [(kernel, grid, threads)]. A step is a function
    of `Steps` and its arguments: ("gemm", True, 512, 4096, 4096). want="orders":
    [(M tiles, N tiles, numbered per XCD, numbered along N)] of tile GEMMs."""
    with tempfile.TemporaryDirectory() as d:
        stub = os.path.join(d, "libhipstub.so")
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", stub, os.path.join(HERE, "hip_stub.c")],
                       check=True)
        r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, want], input=json.dumps(steps),
                           capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout)


def kernel(mangled):
    """(name, [template arguments]) of a mangled kernel name (integral ones)."""
    name = re.search(r"\d+((?:gemm|attn)_[a-z0-9_]+?_kernel)", mangled)
    return (name.group(1) if name else mangled,
            [int(v) for v in re.findall(r"L[ib](\d+)E", mangled[name.end():] if name else "")])


class Steps:
    """The steps, in the process that loaded the stand-in first."""

    def __init__(self, stub):
        self.stub = stub
        torch = types.ModuleType("torch")  # layerops uses it for tensors only
        torch.Tensor = type("Tensor", (), {})
        sys.modules["torch"] = torch
        sys.path.insert(0, HERE)
        from pkg import layerops
        self.L = layerops()

    def order(self, address):
        """The tile counts and orders in a tile GEMM's argument (GemmArgs)."""
        c, p, i = ctypes, ctypes.c_void_p, ctypes.c_int

        class Args(c.Structure):
            _fields_ = [("A", p), ("lda", i), ("a_scale", p), ("W", p), ("M", i), ("N", i), ("K", i), ("I", i),
                        ("ep", self.L.GemmEpilogue), ("partials", p), ("mt", i), ("nt", i), ("vec_out", c.c_bool),
                        ("xcd_order", c.c_bool), ("n_major", c.c_bool)]

        a = Args.from_address(address)
        return a.mt, a.nt, a.xcd_order, a.n_major

    def _ep(self, n):
        return self.L.GemmEpilogue(1.0, 1.0, 1.0, n, n, ADDR, ADDR, ADDR, 1.0, n)

    def gemm(self, fp8, m, n, k, out=0):
        if fp8:
            self.L.call("granite4_gemm_fp8", out, ADDR, k, ADDR, ADDR, m, n, k, self._ep(n))
        else:
            self.L.call("granite4_prefill_gemm", out, ADDR, k, ADDR, m, n, k, self._ep(n), None, 0)

    def gemm_swiglu(self, m, i, k):
        self.L.call("granite4_gemm_fp8_swiglu", ADDR, k, ADDR, ADDR, m, i, k, 1.0, 1.0, ADDR, None, None, ADDR)

    def prefill_attn(self, rows, base, window=0, hk=8, bits=8):
        self.L.call("granite4_prefill_attn", ADDR, rows, 4 * hk, hk, 128, 1 / 128, ADDR, ADDR, ADDR, ADDR, bits,
                    128, 1 << 16, base, ADDR, window, ADDR)

    def multi_step(self, hidden, inter, hq, hk, rows, fp8):
        """granite4_decode_step_multi of one layer, q|k|v one block."""
        L, up = self.L, lambda n: ADDR + n
        y = L.DecodeLayer()
        for f, _ in L.DecodeLayer._fields_:
            setattr(y, f, 1.0 if f in ("sq", "sk", "sv", "so", "sg", "su", "sd") else ADDR)
        y.wk = up(hq * 128 * hidden)
        y.wv = up((hq + hk) * 128 * hidden)
        y.wu = up(inter * hidden)
        m = L.DecodeModel(1, hidden, inter, hq, hk, 1024, 1e-5, 1.0, 1.0, 0.1, ADDR, (L.DecodeLayer * 1)(y), ADDR,
                          ADDR, 1.0, ADDR, ADDR, 1024, 8, 128, 1024)
        b = L.BatchBuffers(16, *[ADDR] * 12)
        L._check(L._lib.granite4_decode_step_multi(m, b, ADDR, rows, int(fp8), None, None), "multi_step")

    def fail_pool_create(self, n):
        self.stub.stub_fail_pool_create(n)

    def capturing(self, on):
        self.stub.stub_capturing(on)


def _child():
    stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    stub.stub_name.restype = ctypes.c_char_p
    stub.stub_arg.restype = ctypes.c_void_p
    s, out = Steps(stub), []
    for name, *args in json.load(sys.stdin):
        stub.stub_reset()
        getattr(s, name)(*args)
        got = []
        for i in range(stub.stub_launches()):
            g = (ctypes.c_uint * 4)()
            stub.stub_grid(i, g)
            got.append(s.order(stub.stub_arg(i)) if sys.argv[2] == "orders" else
                       (stub.stub_name(i).decode(), list(g[:3]), g[3]))
        assert stub.stub_pool_allocs() == stub.stub_pool_frees()
        out.append(got)
    print(json.dumps(out))


if __name__ == "__main__":
    _child()
