"""Records the launches of the C ABI's calls on the host, for test_launch_shapes.py: imported by a process without
torch, whose HIP runtime is tests/cpp/launch_recorder.cpp."""
import ctypes


class Desc(ctypes.Structure):
    """tvdcn_conv_desc of include/tvdcn_hip.h"""
    _fields_ = [("dim", ctypes.c_int32), ("transposed", ctypes.c_int32), ("dtype", ctypes.c_int32),
                ("flags", ctypes.c_int32), ("batch", ctypes.c_int64), ("in_channels", ctypes.c_int64),
                ("out_channels", ctypes.c_int64), ("groups", ctypes.c_int64), ("offset_groups", ctypes.c_int64),
                ("mask_groups", ctypes.c_int64), ("in_size", ctypes.c_int64 * 3), ("kernel", ctypes.c_int64 * 3),
                ("stride", ctypes.c_int64 * 3), ("padding", ctypes.c_int64 * 3), ("dilation", ctypes.c_int64 * 3),
                ("output_padding", ctypes.c_int64 * 3), ("mask_scale", ctypes.c_double)]


def _desc(p):
    d = Desc(dim=p["dim"], transposed=int(p["transposed"]), dtype=p["dtype"], flags=p["flags"], batch=p["batch"],
             in_channels=p["cin"], out_channels=p["cout"], groups=p["groups"], offset_groups=p["og"],
             mask_groups=p["mg"], mask_scale=2.0)
    for i in range(3):
        d.in_size[i] = d.kernel[i] = d.stride[i] = d.dilation[i] = 1
    for i in range(p["dim"]):
        d.in_size[i], d.kernel[i] = p["size"][i], p["kernel"][i]
        d.stride[i] = p["stride"][i] if isinstance(p["stride"], list) else p["stride"]
        d.padding[i], d.dilation[i] = p["padding"], p["dilation"]
        d.output_padding[i] = p["out_pad"]
    return d


def record(recorder_path, lib_path, problems):
    rec = ctypes.CDLL(recorder_path, mode=ctypes.RTLD_GLOBAL)   # ahead of the HIP runtime that the library links
    rec.recorded_name.restype = ctypes.c_char_p
    lib = ctypes.CDLL(lib_path)
    lib.tvdcn_last_error.restype = ctypes.c_char_p
    vp = ctypes.c_void_p
    for name, n in (("forward", 7), ("backward", 11)):
        getattr(lib, f"tvdcn_deform_conv_{name}").argtypes = [ctypes.POINTER(Desc)] + [vp] * n + [ctypes.c_size_t, vp]
        size = getattr(lib, f"tvdcn_deform_conv_{name}_workspace_size")
        size.argtypes, size.restype = [ctypes.POINTER(Desc)], ctypes.c_size_t

    def result(status):
        out = []
        for i in range(rec.recorded_launches()):
            v = (ctypes.c_uint32 * 7)()
            rec.recorded_shape(i, v)
            out.append((rec.recorded_name(i).decode(), list(v[:3]), list(v[3:6])))
        rec.recorded_clear()
        return {"status": status, "error": lib.tvdcn_last_error().decode() if status else "", "launches": out}

    results = []
    for p in problems:
        d = _desc(p)
        x, w, o, m, b, y, gx, gw, go, gm, gb, ws = (vp((i + 1) << 40) for i in range(12))
        if not p["og"]:
            o = go = vp(0)
        if not p["mg"]:
            m = gm = vp(0)
        if not p["bias"]:
            b = gb = vp(0)
        n = lib.tvdcn_deform_conv_forward_workspace_size(ctypes.byref(d))
        st = lib.tvdcn_deform_conv_forward(ctypes.byref(d), x, w, o, m, b, y, ws, n, None)
        r = {"forward": result(st)}
        n = lib.tvdcn_deform_conv_backward_workspace_size(ctypes.byref(d))
        st = lib.tvdcn_deform_conv_backward(ctypes.byref(d), y, x, w, o, m, gx, gw, go, gm, gb, ws, n, None)
        r["backward"] = result(st)
        results.append(r)
    return results
