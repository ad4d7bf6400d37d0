"""Runs calls on one stager against the recording HIP runtime and prints, as
JSON, the operations each call enqueued and which earlier ones they follow.

usage: calls.py RECORDER LIBRARY CALL...
A CALL is KIND:LAYERS_PER_CHUNK:STREAM[:HOST], with KIND pack, unpack or trip,
STREAM a letter and HOST pinned (the default) or pageable; "capture:STREAM"
and "end:STREAM" start and end a stream's capture.  A KIND of pack-null,
unpack-null, inline-pack-null, inline-unpack-null, trip-null-src or
trip-null-dst passes no page ids; its status is printed."""
import ctypes
import json
import sys

L, N, PAGE = 6, 5, 4096
BASE = 1 << 36


def main(recorder, library, *calls):
    rec = ctypes.CDLL(recorder, ctypes.RTLD_GLOBAL)
    rec.rec_name.restype = ctypes.c_char_p
    vp = ctypes.c_void_p
    rec.rec_pinned.argtypes = [vp, ctypes.c_int64]
    rec.rec_capture.argtypes = [vp, ctypes.c_int]
    rec.rec_stream_follows.argtypes = [vp, ctypes.c_int]
    lib = ctypes.CDLL(library)
    lib.pace_kv_last_error.restype = ctypes.c_char_p
    i64 = ctypes.c_int64
    size = L * N * PAGE
    pinned, pageable = BASE, 2 * BASE
    rec.rec_pinned(pinned, size)
    layers = (vp * L)(*[3 * BASE + l * 64 * PAGE for l in range(L)])
    ids = vp(4 * BASE)
    stager = vp()
    assert lib.pace_kv_stager_create(i64(-(-size // 256) * 256), 3, ctypes.byref(stager)) == 0
    out, status = [], []
    for call in calls:
        kind, *rest = call.split(":")
        if kind in ("capture", "end"):
            rec.rec_capture(5 * BASE + ord(rest[0]), kind == "capture")
            continue
        k, stream = int(rest[0]), vp(5 * BASE + ord(rest[1]))
        host = vp(pageable if rest[2:] == ["pageable"] else pinned)
        first = rec.rec_count()
        pool = (layers, L, i64(64), None if "null" in kind else ids, i64(N), i64(PAGE), k)
        suffix = "_inline" if kind.startswith("inline") else ""
        if "unpack" in kind:
            rc = getattr(lib, "pace_kv_unpack_from_host" + suffix)(stager, host, *pool, None, stream)
        elif "pack" in kind:
            rc = getattr(lib, "pace_kv_pack_to_host" + suffix)(stager, *pool, host, None, stream)
        else:
            src, dst = (None if kind == f"trip-null-{side}" else ids for side in ("src", "dst"))
            rc = lib.pace_kv_roundtrip(stager, layers, i64(64), src, layers, i64(64), dst, L, i64(N), i64(PAGE), k,
                                       host, i64(size), None, stream)
        if "null" in kind:
            status.append(rc)
        else:
            assert rc == 0, (call, lib.pace_kv_last_error())
        ops = range(first, rec.rec_count())
        out.append([{"op": o, "name": rec.rec_name(o).decode(), "after": [e for e in range(o) if rec.rec_follows(o, e)],
                     "joined": bool(rec.rec_stream_follows(stream, o))} for o in ops])
    assert lib.pace_kv_stager_destroy(stager) == 0
    print(json.dumps({"calls": out, "status": status, "unwaited": rec.rec_unwaited_at_free()}))


main(*sys.argv[1:])
