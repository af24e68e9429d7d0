"""Runs the library's host code without a GPU, in a process of its own: the
HIP calls go to host_hip.cpp (kernels do not run).  Imported by the programs
that the tests of test_host_calls.py start."""
import ctypes
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LAUNCH = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_uint32,
                          ctypes.POINTER(ctypes.c_void_p))
REFUSE = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_size_t, ctypes.c_int)
D2H = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_size_t)

hip = ctypes.CDLL(os.environ["HOST_HIP"], mode=ctypes.RTLD_GLOBAL)
hip.host_hip_room.restype = ctypes.c_longlong
hip.host_hip_room.argtypes = [ctypes.c_void_p]
hip.host_hip_live_bytes.restype = ctypes.c_longlong
hip.host_hip_new_limit.argtypes = [ctypes.c_size_t]
_keep = []


def hooks(launch=None, refuse=None, d2h=None):
    h = (LAUNCH(launch) if launch else LAUNCH(), REFUSE(refuse) if refuse else REFUSE(),
         D2H(d2h) if d2h else D2H())
    _keep.append(h)
    hip.host_hip_hooks(*h)


def pointer(args, k, offset=0):
    """The pointer at `offset` bytes into kernel argument k."""
    return ctypes.c_void_p.from_address(args[k] + offset).value


def buffer(shape):
    """An array that stands in for device memory."""
    a = np.zeros(shape)
    return a, a.ctypes.data


def lib():
    from mdff_amd import _lib
    L = ctypes.CDLL(_lib.LIB_PATH)
    for name, (res, args) in _lib.PROTOTYPES.items():
        fn = getattr(L, name)
        fn.restype, fn.argtypes = res, args
    return L


dp = ctypes.POINTER(ctypes.c_double)
ip = ctypes.POINTER(ctypes.c_int32)


def create(L, s):
    h = ctypes.c_void_p()
    A = np.ascontiguousarray(np.asarray(s.A, float).reshape(-1, order="F"))
    it = np.ascontiguousarray(s.itype, np.int32)
    st = L.mdffgpu_create(ctypes.byref(s.params), it.ctypes.data_as(ip), A.ctypes.data_as(dp),
                          ctypes.byref(h))
    return st, h


def engforce_device(L, h, r, itime=1):
    from mdff_amd.params import MdffEnergies
    pos = np.ascontiguousarray(r.T)
    f = np.zeros_like(pos)
    en = MdffEnergies()
    return L.mdffgpu_engforce_device(h, pos.ctypes.data, itime, f.ctypes.data, None, None, None,
                                     ctypes.byref(en), None)


def engforce(L, h, r, itime=1):
    from mdff_amd.params import MdffEnergies
    x = [np.ascontiguousarray(r[:, a]) for a in range(3)]
    f = [np.zeros(len(r)) for _ in range(3)]
    en = MdffEnergies()
    d = lambda a: a.ctypes.data_as(dp)
    return L.mdffgpu_engforce(h, *map(d, x), itime, *map(d, f), None, None, None, None,
                              ctypes.byref(en))


def melt(n, pim):
    """A silica system of n atoms at random positions (no kernel runs)."""
    from mdff_amd import configs as C
    s = C.silica(20, 40, seed=8, rc=4.0, kmax=3, pim=pim)
    L = max(8.1, (13.0 * n) ** (1.0 / 3.0))
    s.params.natm = n
    A = L * np.eye(3)
    itype = np.repeat([1, 2], [n // 3, n - n // 3]).astype(np.int32)
    return C.System(s.params, itype, A, L * np.random.default_rng(n).random((n, 3)), s.name, {})


def efg(L, h, r):
    from mdff_amd import params as P
    x = [np.ascontiguousarray(r[:, a]) for a in range(3)]
    out = np.zeros(9 * len(r))
    en = P.MdffEnergies()
    d = lambda a: a.ctypes.data_as(dp)
    return L.mdffgpu_efg(h, ctypes.byref(P.efg_opts("ewald")), *map(d, x), None, d(out),
                         ctypes.byref(en))
