"""The library's own choice of a route for a shape (ozablas_amd/csrc/plan_host.cpp), read on the host through its
internal symbols, so that a test can hold each of its cases to the route it is there for."""
import ctypes as C


class Dims(C.Structure):
    _fields_ = [(n, C.c_int64) for n in ("M", "N", "K", "Mp", "Np", "Kp")] + [("S", C.c_int)]


class S2Plan(C.Structure):
    _fields_ = [("edge", C.c_int), ("parts", C.c_int), ("kts", C.c_int), ("whole", C.c_int64)]


class S1Plan(C.Structure):
    _fields_ = [("edge", C.c_int), ("parts", C.c_int * 20), ("planes", C.c_int)]


def _call(name, restype, *args):
    import ozablas_amd as oz

    f = oz.lib[name]
    f.restype = restype
    f.argtypes = [type(a) for a in args]
    return f(*args)


def _dims(M, N, K, S):
    return _call("_ZN3oza9make_dimsEmmmi", Dims, C.c_size_t(M), C.c_size_t(N), C.c_size_t(K), C.c_int(S))


def s2(M, N, K, S):
    """Scheme II: edge, parts and whole of the plan, its items (parts counted) and whether it takes four slots."""
    d = _dims(M, N, K, S)
    p = _call("_ZN3oza12scheme2_planERKNS_4DimsE", S2Plan, C.pointer(d))
    deep = _call("_ZN3oza12s2_deep_ringERKNS_4DimsERKNS_6S2PlanE", C.c_bool, C.pointer(d), C.pointer(p))
    items = -(-M // p.edge) * -(-N // p.edge) * S
    if p.parts > 1:
        items += (p.parts - 1) * (items - p.whole)
    short = p.parts > 1 and p.parts * p.kts != d.Kp // 128  # the last part is shorter
    return dict(edge=p.edge, parts=p.parts, whole=p.whole if p.parts > 1 else items, items=items, deep=deep, short=short)


def s1(M, N, K, S):
    """Scheme I: edge, planes (more than S: groups in parts) and whether its items come from the work counters."""
    p = _call("_ZN3oza12scheme1_planERKNS_4DimsE", S1Plan, C.pointer(_dims(M, N, K, S)))
    tiles = -(-M // p.edge) * -(-N // p.edge)
    return dict(edge=p.edge, planes=p.planes, dynamic=p.edge == 256 and tiles >= 64 and tiles * p.planes >= 512)
