"""What a context's one-launch solves (csrc/group.hip) did, through the
library's test aids."""
import ctypes as C

from mhfem_amd import capi

HOLD = ("memory", "registers", "lds")


def _call(name, s, *args):
    fn = getattr(capi.lib(), name)
    fn.restype = C.c_int
    assert fn(C.c_void_p(s.ctx), *args) == 0, name


def info(s):
    v = (C.c_longlong * 10)()
    _call("mhfem_internal_group_info", s, v, C.c_int(10))
    return dict(total=v[0], threads=v[1], hold=HOLD[v[2]], launches=v[3], gave_up=v[4], cooldown=v[5], planes=v[6],
                iterations=v[7], neighbours=v[8], remote=v[9])


def launched(s, off=True):
    """The context iterates by launches also where one launch would do."""
    _call("mhfem_internal_group_off", s, C.c_int(off))


def wait_bound(s, ticks):
    _call("mhfem_internal_group_wait", s, C.c_ulonglong(ticks))


def iterated_in_one_launch(s):
    """At least one solve did, and none gave up."""
    i = info(s)
    return i["total"] > 0 and i["launches"] > 0 and i["gave_up"] == 0
