"""Runs library calls on the fake runtime and prints what they did: argv is the
fake runtime, the library and a JSON list of steps.  A step is ["capture", 0/1],
["room", bytes or null] or [entry point, n, m, tokens, {options}]; a call's
result is its status and the lines of the runtime's log (one JSON value a
step)."""
import ctypes
import json
import sys

fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
fake.fake_log.restype = ctypes.c_char_p
fake.fake_set_room.argtypes = [ctypes.c_size_t]
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "f16": (1, 2), "q4_0_col": (32, 18)}
_p, _z = ctypes.c_void_p, ctypes.c_size_t
out = []
for step in json.loads(sys.argv[3]):
    if step[0] == "capture":
        fake.fake_set_capturing(step[1])
        out.append(None)
    elif step[0] == "room":
        fake.fake_set_room(2 ** 64 - 1 if step[1] is None else step[1])
        out.append(None)
    else:
        kind, n, m, tokens = step[:4]
        opt = step[4] if len(step) > 4 else {}
        elems, size = BLOCK[kind.replace("_noalloc", "")]
        w_len = -(-n * m // elems) * size + opt.get("extra", 0)
        name = {"q4_0_noalloc": "hypno_hip_matmul_q4_0_dev_noalloc"}.get(
            kind, f"hypno_hip_matmul_{kind}_dev")
        fn = getattr(lib, name)
        fn.argtypes = [_p, _p, _z, _p, _p, _z, _z, _z, _p]
        # addresses of nothing: y, w, x apart
        st = fn(1 << 40, (2 << 40) + opt.get("w_off", 0), w_len, (3 << 40) + opt.get("x_off", 0),
                None, n, m, tokens, opt.get("stream", 0))
        out.append([st, fake.fake_log().decode().splitlines()])
print(json.dumps(out))
