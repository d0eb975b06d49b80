"""The library's host code on the CPU against the stand-in HIP runtime (fakehip.c) with kernel launches
recorded, not executed: what is launched, and what the host does within a given amount of device memory.

Test infrastructure only. Create a HostSim before the first use of cgfdm_amd.solver in the process."""
import ctypes
import os
import re
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path[:0] = [HERE, os.path.join(ROOT, "cgfdm3d-eqr-sc_amd")]
import simgpu  # noqa: E402


class HostSim:
    def __init__(self, limit=1 << 40):
        self.limit, self.used, self.peak, self.bufs, self.launches = limit, 0, 0, {}, []
        self.lib = ctypes.CDLL(simgpu.build_fakehip(), mode=ctypes.RTLD_GLOBAL)
        A = ctypes.CFUNCTYPE(ctypes.c_uint64, ctypes.c_uint64)
        F = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_uint64)
        L = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, *([ctypes.c_uint32] * 6), ctypes.POINTER(ctypes.c_void_p),
                             ctypes.c_uint64)
        self._cbs = (A(self._alloc), F(self._free), L(self._launch))
        self.lib.fakehip_set_callbacks(*self._cbs)

    def _alloc(self, n):
        if self.used + n > self.limit:
            return 0
        b = ctypes.create_string_buffer(int(n) + 256)
        a = (ctypes.addressof(b) + 255) // 256 * 256
        self.bufs[a] = (b, int(n))
        self.used += int(n)
        self.peak = max(self.peak, self.used)
        return a

    def _free(self, a):
        self.used -= self.bufs.pop(a)[1]
        return 0

    def _launch(self, name, gx, gy, gz, bx, by, bz, args, shmem):
        m = re.match(r"_ZN2(?:cg|aw)\d+([a-z0-9_]+?)I", name.decode()) or re.match(r"_ZN2(?:cg|aw)\d+([a-z0-9_]+)E", name.decode())
        self.launches.append((m.group(1) if m else name.decode(), (gx, gy, gz)))
        return 0

    def names(self):
        """Names of the kernels launched since the last call."""
        out = [n for n, _ in self.launches]
        self.launches.clear()
        return out
