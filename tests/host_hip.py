"""The library on a machine without a GPU: hip_stand_in.c takes the place of
the HIP runtime in a child process, so that a test sees which kernels a call
launches, what it allocates and what it does when memory is short.

``run(name, *args)`` calls the function ``name`` of the calling test module in
such a process and returns its (JSON) result; in there, ``HostHip`` is the
library on the stand-in."""
import ctypes as C
import json
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def build(folder):
    """Compile the stand-in into ``folder``; its path."""
    out = os.path.join(str(folder), "hip_stand_in.so")
    subprocess.run(["gcc", "-std=c11", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", out, os.path.join(HERE, "hip_stand_in.c")],
                   check=True)
    return out


def run(module_file, stand_in, name, *args):
    code = (f"import sys, json; sys.path[:0] = {[ROOT, HERE]!r}\n"
            f"import host_hip, {os.path.basename(module_file)[:-3]} as m\n"
            f"print(json.dumps(m.{name}(host_hip.HostHip({stand_in!r}), *json.loads(sys.argv[1]))))")
    r = subprocess.run([sys.executable, "-c", code, json.dumps(args)], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.splitlines()[-1])


class HostHip:
    def __init__(self, stand_in):
        self.s = C.CDLL(stand_in, mode=C.RTLD_GLOBAL)     # before the library
        self.s.standin_live.restype = self.s.standin_allocation.restype = C.c_size_t
        self.s.standin_limit.argtypes = [C.c_size_t]
        self.s.standin_launch.restype = C.c_char_p
        from random_amd import _lib
        self.lib = _lib.lib()
        # an address for arrays that no kernel will read
        self.any = C.cast(C.create_string_buffer(4096), C.c_void_p).value & ~0xff

    def limit(self, nbytes=None):
        self.s.standin_limit(2 ** 64 - 1 if nbytes is None else nbytes)

    def live(self):
        return self.s.standin_live()

    def plan(self, cfg, ns, dt, vel):
        from random_amd import _lib
        h, c = C.c_void_p(), cfg.to_c()
        _lib.check(self.lib.ktm_plan_create(C.byref(h), C.byref(c), ns, dt, vel.shape[2], dt,
                                            vel.ctypes.data_as(C.c_void_p)), "ktm_plan_create")
        return h

    def call(self, name, *args):
        """(status, launches, allocated bytes) of one call; a launch of a kernel
        of this library is (kernel, its integer template arguments, grid,
        workgroup, LDS)."""
        self.s.standin_clear()
        st = getattr(self.lib, name)(*args)
        out = []
        for i in range(self.s.standin_launches()):
            d = (C.c_uint32 * 7)()
            sym = self.s.standin_launch(i, d).decode()
            m = re.match(r"_Z(\d+)(k_.*)", sym)
            if not m:
                continue                                  # the sort's
            n = int(m.group(1))
            t = [int(v) for v in re.findall(r"L[ib](\d+)E", m.group(2)[n:])]
            out.append((m.group(2)[:n], t, list(d[0:3]), list(d[3:6]), d[6]))
        return st, out, [self.s.standin_allocation(i) for i in range(self.s.standin_allocations())]

    def migrate(self, plan, ntr, accum, job=-1, dtype=0, mode=1):
        return self.call("ktm_migrate_block", plan, self.any, dtype, mode, self.any, ntr, accum, job,
                         self.any, self.any, self.any, None, None)

    def demigrate(self, plan, ntr):
        return self.call("ktm_demigrate", plan, self.any, self.any, ntr, self.any, None)
