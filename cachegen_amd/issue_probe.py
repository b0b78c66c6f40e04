"""ctypes binding of lib/libcachegen_probe.so (csrc/issue_probe.hip): how fast a SIMD of this GPU
issues vector instructions and at which engine clock.  A measuring tool for bench.py and the
profiles, not part of the codec; nothing under serde/ or codec.py uses it."""
import ctypes

from .build import PROBE_LIBRARY

_handle = None

CHEAP, FULL, DECODER_SYMBOL = 0, 1, 2


def lib():
    global _handle
    if _handle is None:
        try:
            h = ctypes.CDLL(PROBE_LIBRARY)
        except OSError as e:
            raise RuntimeError("calibration probe not built (%s): run cachegen_amd.build.build_probe()" % e)
        h.cg_probe_issue_rate.restype = ctypes.c_int
        h.cg_probe_issue_rate.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_double)]
        h.cg_probe_clock_start.restype = ctypes.c_int
        h.cg_probe_clock_start.argtypes = [ctypes.c_int, ctypes.c_void_p]
        h.cg_probe_clock_result.restype = ctypes.c_int
        h.cg_probe_clock_result.argtypes = [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_double)]
        h.cg_probe_op.restype = h.cg_probe_chain.restype = ctypes.c_char_p
        h.cg_probe_op.argtypes = h.cg_probe_chain.argtypes = [ctypes.c_int]
        h.cg_probe_pair_start.argtypes = [ctypes.c_int] * 4
        h.cg_probe_pair_wait.argtypes = [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_double)]
        h.cg_probe_chain_cycles.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_double)]
        h.cg_probe_pci.argtypes = [ctypes.c_char_p, ctypes.c_int]
        _handle = h
    return _handle


def issue_rate(kind, iters=2048):
    """(ns per wave64 instruction per SIMD with 8 wavefronts resident, engine clock in MHz)."""
    ns, mhz = ctypes.c_double(), ctypes.c_double()
    rc = lib().cg_probe_issue_rate(kind, iters, ctypes.byref(ns), ctypes.byref(mhz))
    if rc:
        raise RuntimeError("cg_probe_issue_rate: hipError %d" % rc)
    return ns.value, mhz.value


def calibrate(iters=2048):
    """Cycles a SIMD takes per wave64 instruction of the cheap class, of the full-rate class and of
    the decoder's own instruction sequence, with the engine clock each was measured at."""
    out = {}
    for name, kind in (("cheap", CHEAP), ("full", FULL), ("decoder_symbol", DECODER_SYMBOL)):
        ns, mhz = issue_rate(kind, iters)
        out[name] = {"ns_per_instruction": round(ns, 4), "clock_mhz": round(mhz, 1), "cycles_per_instruction": round(ns * mhz * 1e-3, 3)}
    return out


def clock_window_start(microseconds, stream):
    """Queue the one-wavefront clock sampler on `stream` (a raw hipStream_t) for about that long."""
    rc = lib().cg_probe_clock_start(int(microseconds), ctypes.c_void_p(stream))
    if rc:
        raise RuntimeError("cg_probe_clock_start: hipError %d" % rc)


def clock_window_result():
    """(engine clock in MHz averaged over the sampler's window, window length in microseconds);
    call after the sampler's stream has been synchronized."""
    mhz, us = ctypes.c_double(), ctypes.c_double()
    rc = lib().cg_probe_clock_result(ctypes.byref(mhz), ctypes.byref(us))
    if rc:
        raise RuntimeError("cg_probe_clock_result: hipError %d" % rc)
    return mhz.value, us.value


def _check(rc, what):
    if rc:
        raise RuntimeError("%s: hipError %d" % (what, rc))


def _names(name):
    out = []
    while name(len(out)):
        out.append(name(len(out)).decode())
    return out


def ops():
    """The instructions that `pair` takes by number."""
    return _names(lib().cg_probe_op)


def _pair_wait():
    ns, mhz = ctypes.c_double(), ctypes.c_double()
    _check(lib().cg_probe_pair_wait(ctypes.byref(ns), ctypes.byref(mhz)), "cg_probe_pair_wait")
    return ns.value, mhz.value


def pair(a, b, iters=256):
    """Cycles a full SIMD takes for one instruction `a` and one `b`, issued a a b b."""
    for launches in (2, 8):                                    # the first brings the clock up
        _check(lib().cg_probe_pair_start(a, b, iters, launches), "cg_probe_pair_start")
        ns, mhz = _pair_wait()
    return 2.0 * ns * mhz * 1e-3


def chains():
    """{chain: cycles of a link} for one wavefront alone on its compute unit."""
    out = {}
    for i, name in enumerate(_names(lib().cg_probe_chain)):
        cycles = ctypes.c_double()
        _check(lib().cg_probe_chain_cycles(i, ctypes.byref(cycles)), "cg_probe_chain_cycles")
        out[name] = cycles.value
    return out


def power_file():
    """The file in which the driver reports this card's power, in microwatts; None if it does not."""
    import glob
    address = ctypes.create_string_buffer(32)
    _check(lib().cg_probe_pci(address, 32), "cg_probe_pci")
    where = "/sys/bus/pci/devices/%s/hwmon/hwmon*/" % address.value.decode().lower()
    return (glob.glob(where + "power1_average") + glob.glob(where + "power1_input") + [None])[0]


def power(op, path, seconds=0.8, iters=512):
    """(W, ns an instruction, engine clock in MHz) of a card that does nothing else than `op` for about that long."""
    import time
    _check(lib().cg_probe_pair_start(op, op, iters, 20), "cg_probe_pair_start")
    ns, _ = _pair_wait()
    launches = max(1, int(seconds * 1e9 / (ns * 32 * iters * 64)))             # 8 wavefronts a SIMD, 4 rounds
    _check(lib().cg_probe_pair_start(op, op, iters, launches), "cg_probe_pair_start")
    time.sleep(seconds / 2)
    watts = []
    for _ in range(12):
        watts.append(int(open(path).read()) * 1e-6)
        time.sleep(seconds / 48)
    ns, mhz = _pair_wait()
    return sum(watts) / len(watts), ns, mhz


def details():
    """What the figures in the documentation come from, as text: pairs of instructions, chains, energy."""
    import torch
    simds = torch.cuda.get_device_properties(0).multi_processor_count * 4
    names = ops()
    print("cycles of a full SIMD (8 wavefronts) for one instruction of the row and one of the column, issued two and two")
    width = max(map(len, names)) + 1
    print(" " * width + " ".join("%5d" % i for i in range(1, len(names) - 1)))
    for i in range(1, len(names) - 1):                         # without s_nop and the LDS read
        print("%-*s" % (width, names[i]) + " ".join("%5.1f" % pair(i, j) for j in range(1, i + 1)) + "   (%d)" % i, flush=True)
    print("cycles of a dependent link, one wavefront alone on its compute unit")
    for name, cycles in chains().items():
        print("%-34s %6.1f" % (name, cycles))
    path = power_file()
    if path is None:
        print("no power reading on this machine")
        return
    try:
        print("the card's power limit: %.0f W" % (int(open(path.rsplit("/", 1)[0] + "/power1_cap").read()) * 1e-6))
    except OSError:
        pass
    print("one instruction in a loop on every SIMD: card's power, and energy a wave64 instruction above s_nop's")
    idle = None
    for i, name in enumerate(names):
        watts, ns, mhz = power(i, path)
        idle = watts if idle is None else idle
        print("%-16s %6.0f W  %6.3f ns  %5.0f MHz  %6.2f nJ" % (name, watts, ns, mhz, (watts - idle) * ns / simds), flush=True)


if __name__ == "__main__":
    import json
    import sys
    if sys.argv[1:] == ["--details"]:
        details()
    else:
        print(json.dumps(calibrate(), indent=1))
