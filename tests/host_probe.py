"""Subprocess helper of tests/test_host_paths.py (not collected by pytest): loads the stub HIP
runtime (hip_stub.c, built by the test) ahead of libtaskops.so, without torch, and runs the
steps given as JSON on stdin.  A step is {"call": symbol, "types": "pifl...", "args": [...]} or
{"set": name, "args": [...]}; for each it prints the return code and the stub's record.

    python tests/host_probe.py STUB.so LIBTASKOPS.so < steps.json
"""
import ctypes
import json
import sys

TYPES = {"p": ctypes.c_void_p, "i": ctypes.c_int32, "l": ctypes.c_int64, "f": ctypes.c_float}


def main() -> None:
    stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    stub.stub_log.restype = ctypes.c_char_p
    lib = ctypes.CDLL(sys.argv[2])
    out = []
    for step in json.load(sys.stdin):
        stub.stub_clear()
        if "set" in step:
            getattr(stub, "stub_set_" + step["set"])(*step["args"])
            rc = 0
        else:
            fn = getattr(lib, step["call"])
            fn.argtypes = [TYPES[t] for t in step["types"]]
            rc = fn(*step["args"])
        out.append({"rc": rc, "log": stub.stub_log().decode().splitlines()})
    print(json.dumps(out))


if __name__ == "__main__":
    main()
