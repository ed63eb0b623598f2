"""Performance cases: the work a program gives this library, at the sizes it meets in use.

Each case is a dict of plain values; its `kind` names the path:

  call          one codeword through the Python classes (host buffers): encode, then repair of a damaged copy
  rs256_encode  RS256 parity of a batch resident in HBM
  rs256_repair  RS256 repair of a damaged batch resident in HBM
  rsi16_encode  RSi16 parity of a batch resident in HBM
  rsi16_repair  RSi16 repair of a damaged batch resident in HBM
  mixed         mixed-size work lists (one RS256 plan, one RSi16 plan): encode, then repair of damaged copies
  circ16        a file buffer through CIRC16 as `par backup` and `par repair` take it (host buffers)

Repairs work in place, so each pass first restores the damaged codewords from a pristine copy, on the codec's
stream, as a program does that keeps what it received.

All outputs are symbols, bytes and status codes of exact finite-field arithmetic.
"""
import functools

import numpy as np
import torch

import libffrs_amd
from libffrs_amd import capi, par
from libffrs_amd.par.opt import choose_geometry

MIXED_RS256_ECC = (2, 4, 8, 16, 32, 64)
MIXED_RSI16_N = (64, 256, 1024)
MIXED_RSI16_ECC = (8, 16, 32)


def listed():
    return [
        # The reference's own way of working: one codeword per call. Latency and launches are all of it.
        {"name": "call_rs256_ecc32", "kind": "call", "field": "rs256", "k": 223, "ecc": 32, "errors": 16},
        # The plain small batch of the benchmark: 4,096 messages, a few microseconds of device work.
        {"name": "rs256_repair_ecc8_small", "kind": "rs256_repair", "k": 247, "ecc": 8, "count": 4096, "errors": 4,
         "beyond": 0.0},
        # The benchmark's default workload, RS(255,223) on a million codewords, in both directions;
        # 1% of the damaged codewords are beyond the radius.
        {"name": "rs256_encode_ecc32", "kind": "rs256_encode", "k": 223, "ecc": 32, "count": 1048576},
        {"name": "rs256_repair_ecc32", "kind": "rs256_repair", "k": 223, "ecc": 32, "count": 1048576, "errors": 16,
         "beyond": 0.01},
        # An ordinary batch of an odd shape: a shortened code, parity length no power of two, odd row lengths.
        {"name": "rs256_repair_ecc21_odd", "kind": "rs256_repair", "k": 130, "ecc": 21, "count": 100003, "errors": 10,
         "beyond": 0.01},
        # The benchmark's RSi16 workload: many short blocks, both directions.
        {"name": "rsi16_encode_256_32", "kind": "rsi16_encode", "n": 256, "ecc": 32, "count": 262144},
        {"name": "rsi16_repair_256_32", "kind": "rsi16_repair", "n": 256, "ecc": 32, "count": 262144, "errors": 16,
         "burst": False},
        # Its large-block variant, both directions.
        {"name": "rsi16_encode_4096_256", "kind": "rsi16_encode", "n": 4096, "ecc": 256, "count": 16384},
        {"name": "rsi16_repair_4096_256", "kind": "rsi16_repair", "n": 4096, "ecc": 256, "count": 16384,
         "errors": 128, "burst": False},
        # The serving loop's largest piece of a request: verify + repair of 2,048 par-style blocks, 0-5% of
        # their symbols damaged, half of them in bursts.
        {"name": "rsi16_repair_1024_128", "kind": "rsi16_repair", "n": 1024, "ecc": 128, "count": 2048, "errors": 51,
         "burst": True},
        # The mixed-size batch of the benchmark: ragged lengths, 1,404 + 9 size classes.
        {"name": "mixed_plans", "kind": "mixed", "rs256": 200000, "rsi16": 50000},
        # A 4 MiB file through backup and repair (host buffers, as files are read and written).
        {"name": "circ16_file_4m", "kind": "circ16", "size": 4194304, "lost": 0.02},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("call", "rs256_encode", "rs256_repair", "rs256_repair", "rsi16_encode", "rsi16_repair",
                       "rsi16_repair", "mixed", "circ16"))
    if kind == "call":
        if rng.random() < 0.5:
            ecc = rng.choice((2, 4, 7, 8, 16, 21, 32, 48, 64))
            return {"kind": kind, "field": "rs256", "k": rng.randint(1, 255 - ecc), "ecc": ecc,
                    "errors": rng.randint(0, ecc // 2)}
        ecc = rng.choice((8, 16, 32, 64, 128))
        return {"kind": kind, "field": "rsi16", "k": ecc * rng.randint(1, 1024 // ecc - 1), "ecc": ecc,
                "errors": rng.randint(0, ecc // 2)}
    if kind.startswith("rs256"):
        ecc = rng.choice((2, 4, 8, 8, 16, 32, 32, rng.randint(1, 32), rng.randint(1, 32), rng.randint(33, 64)))
        k = 255 - ecc if rng.random() < 0.4 else rng.randint(1, 255 - ecc)
        most = min(1048576 if ecc <= 32 else 32768, 267386880 // (k + ecc))
        case = {"kind": kind, "k": k, "ecc": ecc, "count": _log_uniform(rng, 4096, most)}
        if kind == "rs256_repair":
            case.update(errors=ecc // 2, beyond=rng.choice((0.0, 0.01)))
        return case
    if kind.startswith("rsi16"):
        ecc = rng.choice((8, 16, 32, 32, 64, 128, 256))
        n = ecc * rng.randint(2, 4096 // ecc) if rng.random() < 0.5 else ecc * 2 ** rng.randint(1, (4096 // ecc).bit_length() - 1)
        most = min(262144, (1 << 30) // (ecc * ecc), 67108864 // n)
        case = {"kind": kind, "n": n, "ecc": ecc, "count": _log_uniform(rng, 512, most)}
        if kind == "rsi16_repair":
            case.update(errors=ecc // 2, burst=rng.random() < 0.5)
        return case
    if kind == "mixed":
        return {"kind": kind, "rs256": _log_uniform(rng, 2000, 200000), "rsi16": _log_uniform(rng, 500, 50000)}
    while True:  # sizes for which the file front end has a geometry
        size = _log_uniform(rng, 16384, 4194304)
        try:
            choose_geometry(size)
            break
        except ValueError:
            continue
    return {"kind": kind, "size": size, "lost": round(0.01 + 0.03 * rng.random(), 4)}


# ---- what a program keeps for its whole life: one context, one codec per shape ----------------


@functools.lru_cache(None)
def _context():
    return capi.Context(0)


@functools.lru_cache(None)
def _rs256(ecc):
    return capi.RS256Codec(_context(), ecc)


@functools.lru_cache(None)
def _rsi16(n, ecc):
    return capi.RSi16Codec(_context(), n, ecc)


@functools.lru_cache(None)
def _host_codec(field, k, ecc):
    return libffrs_amd.RS256(ecc_len=ecc, message_len=k) if field == "rs256" else libffrs_amd.RSi16(k + ecc, ecc)


@functools.lru_cache(None)
def _circ16(size):
    return par.choose_codec(size)


# ---- inputs ------------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _view(t):
    return capi.DeviceBuffer(_context(), t.data_ptr(), t.numel() * t.element_size())


def _damage(value, gen):
    """Another symbol in each place, uniform over the others."""
    if value.dtype == torch.uint8:  # XOR with a non-zero byte
        return value ^ torch.randint(1, 256, value.shape, generator=gen, device="cuda", dtype=torch.uint8)
    v = value.to(torch.int32) & 0xFFFF  # a non-zero offset mod 65537 whose sum is a u16 value
    v = (v + torch.randint(1, 65536, v.shape, generator=gen, device="cuda", dtype=torch.int32)) & 0xFFFF
    return v.to(torch.int16)


def _damage_rows(rows, counts, gen):
    """Damages counts[i] distinct symbols of rows[i], in place."""
    n, most = rows.shape[1], int(counts.max()) if counts.numel() else 0
    step = max(1, (1 << 26) // n)
    for a in range(0, rows.shape[0] if most else 0, step):
        part, c = rows[a:a + step], counts[a:a + step]
        pos = torch.rand(part.shape, generator=gen, device="cuda").topk(most, dim=1, sorted=False).indices
        r, j = (torch.arange(most, device="cuda")[None, :] < c[:, None]).nonzero(as_tuple=True)
        p = pos[r, j]
        part[r, p] = _damage(part[r, p], gen)


def _damage_bursts(rows, share, gen):
    """Damages a `share` of the symbols, half alone and half in runs of 8 to 64, as if rows were one file."""
    flat = rows.view(-1)
    count = int(flat.numel() * share)
    single = torch.randint(0, flat.numel(), (count // 2,), generator=gen, device="cuda")
    runs = max(1, count // 2 // 36)
    start = torch.randint(0, flat.numel() - 64, (runs,), generator=gen, device="cuda")
    length = torch.randint(8, 65, (runs,), generator=gen, device="cuda")
    at = torch.arange(64, device="cuda")
    pos = torch.cat([single, (start[:, None] + at)[at[None, :] < length[:, None]]]).unique()
    flat[pos] = _damage(flat[pos], gen)


def _error_counts(case, count, gen):
    c = torch.randint(0, case["errors"] + 1, (count,), generator=gen, device="cuda")
    n = case["k"] + case["ecc"]
    beyond = int(count * case.get("beyond", 0.0))
    if beyond:
        at = torch.arange(beyond, device="cuda") * count // beyond
        more = torch.randint(1, 5, (beyond,), generator=gen, device="cuda")
        c[at] = (case["ecc"] // 2 + more).clamp(max=n)
    return c.clamp(max=n)


class _State:
    """The buffers of one case; plans are given back with it."""

    plans = ()

    def __del__(self):
        for p in self.plans:
            p.close()


def _prepare_batch(case, seed):
    s, gen, rs256 = _State(), _generator(seed), case["kind"].startswith("rs256")
    ecc, count = case["ecc"], case["count"]
    k = case["k"] if rs256 else case["n"] - ecc
    s.k, s.count, s.rs256 = k, count, rs256
    s.codec = _rs256(ecc) if rs256 else _rsi16(k + ecc, ecc)
    dtype = torch.uint8 if rs256 else torch.int16
    lo, hi = (0, 256) if rs256 else (-32768, 32768)
    msg = torch.randint(lo, hi, (count, k), generator=gen, device="cuda", dtype=dtype)
    par_ = torch.zeros((count, ecc), device="cuda", dtype=dtype)
    torch.cuda.synchronize()
    if rs256:
        s.codec.encode_device(k, _view(msg), count, _view(par_))
    else:
        s.codec.encode_device(_view(msg), count, _view(par_))
    _context().sync()
    s.msg, s.par = msg, par_
    s.v_msg, s.v_par = _view(msg), _view(par_)
    if case["kind"].endswith("encode"):
        s.par = torch.zeros_like(par_)
        s.v_par = _view(s.par)
        return s
    rows = torch.cat([msg, par_], 1)
    if case.get("burst"):
        # up to `errors` symbols per codeword on average; a request has one share, a piece holds several requests
        step = max(1, count // 8)
        shares = torch.rand(8 + 1, generator=gen, device="cuda").tolist()
        for i, a in enumerate(range(0, count, step)):
            if rows[a:a + step].numel() > 64:
                _damage_bursts(rows[a:a + step], shares[i % 9] * min(0.05, case["errors"] / (k + ecc)), gen)
    else:
        _damage_rows(rows, _error_counts({**case, "k": k}, count, gen), gen)
    s.bad_msg, s.bad_par = rows[:, :k].contiguous(), rows[:, k:].contiguous()
    s.status = torch.zeros(count, device="cuda", dtype=torch.uint8)
    s.v_bad_msg, s.v_bad_par, s.v_status = _view(s.bad_msg), _view(s.bad_par), _view(s.status)
    return s


def _offsets(lens):
    return np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.uint64)


def _ragged_damage(s, msg, par_, lens, eccs, moff, eoff, gen):
    """Damages up to ecc / 2 distinct symbols of each listed codeword, uniform over message and parity."""
    dev = lambda a: torch.from_numpy(np.asarray(a, np.int64)).cuda()  # noqa: E731
    lens, eccs, moff, eoff = dev(lens), dev(eccs), dev(moff), dev(eoff)
    width, most = int((lens + eccs).max()), int(eccs.max()) // 2
    step = max(1, (1 << 26) // width)
    at = torch.arange(width, device="cuda")[None, :]
    for a in range(0, len(lens), step):
        k, e = lens[a:a + step], eccs[a:a + step]
        keys = torch.rand((len(k), width), generator=gen, device="cuda")
        pos = keys.masked_fill(at >= (k + e)[:, None], -1.0).topk(min(most, width), dim=1, sorted=True).indices
        c = (torch.rand(len(k), generator=gen, device="cuda") * (e // 2 + 1)).long()
        c = torch.minimum(c, k + e)
        r, j = (torch.arange(pos.shape[1], device="cuda")[None, :] < c[:, None]).nonzero(as_tuple=True)
        p = pos[r, j]
        inside = p < k[r]
        m = moff[a + r[inside]] + p[inside]
        q = eoff[a + r[~inside]] + (p - k[r])[~inside]
        msg[m] = _damage(msg[m], gen)
        par_[q] = _damage(par_[q], gen)


def _prepare_mixed(case, seed):
    s, gen = _State(), _generator(seed)
    rng = np.random.default_rng(case["rs256"])  # the lists' shapes belong to the case, their contents to the seed
    e8 = rng.choice(MIXED_RS256_ECC, case["rs256"])
    k8 = rng.integers(1, 256 - e8)
    n16, e16 = rng.choice(MIXED_RSI16_N, case["rsi16"]), rng.choice(MIXED_RSI16_ECC, case["rsi16"])
    k16 = n16 - e16
    m8, p8, m16, p16 = _offsets(k8), _offsets(e8), _offsets(k16), _offsets(e16)
    s.plan8 = capi.RS256Plan(_context(), e8, k8, m8, p8, graph=True)
    s.plan16 = capi.RSi16Plan(_context(), n16, e16, m16, p16, graph=True)
    s.plans = (s.plan8, s.plan16)
    s.msg = [torch.randint(0, 256, (int(k8.sum()),), generator=gen, device="cuda", dtype=torch.uint8),
             torch.randint(-32768, 32768, (int(k16.sum()),), generator=gen, device="cuda", dtype=torch.int16)]
    s.par = [torch.zeros(int(e8.sum()), device="cuda", dtype=torch.uint8),
             torch.zeros(int(e16.sum()), device="cuda", dtype=torch.int16)]
    torch.cuda.synchronize()
    s.v_msg, s.v_par = [_view(t) for t in s.msg], [_view(t) for t in s.par]
    s.plan8.encode(s.v_msg[0], s.v_par[0])
    s.plan16.encode(s.v_msg[1], s.v_par[1])
    _context().sync()
    s.bad_msg, s.bad_par = [t.clone() for t in s.msg], [t.clone() for t in s.par]
    _ragged_damage(s, s.bad_msg[0], s.bad_par[0], k8, e8, m8, p8, gen)
    _ragged_damage(s, s.bad_msg[1], s.bad_par[1], k16, e16, m16, p16, gen)
    s.fix_msg, s.fix_par = [t.clone() for t in s.bad_msg], [t.clone() for t in s.bad_par]
    s.status = [torch.zeros(case["rs256"], device="cuda", dtype=torch.uint8),
                torch.zeros(case["rsi16"], device="cuda", dtype=torch.uint8)]
    for name in ("bad_msg", "bad_par", "fix_msg", "fix_par", "status"):
        setattr(s, "v_" + name, [_view(t) for t in getattr(s, name)])
    return s


def _prepare_call(case, seed):
    s, rng = _State(), np.random.default_rng(int(seed))
    s.codec = _host_codec(case["field"], case["k"], case["ecc"])
    dtype, size = (np.uint8, 256) if case["field"] == "rs256" else (np.uint16, 65536)
    s.dtype = dtype
    msg = rng.integers(0, size, case["k"]).astype(dtype)
    s.msg = msg.tobytes()
    row = np.concatenate([msg, np.frombuffer(bytes(s.codec.encode(s.msg)), dtype)])
    at = rng.choice(row.size, min(case["errors"], row.size), replace=False)
    row[at] = (row[at].astype(np.int64) + rng.integers(1, size, at.size)) % size
    s.bad_msg, s.bad_par = row[:case["k"]].tobytes(), row[case["k"]:].tobytes()
    return s


def _prepare_circ16(case, seed):
    s, rng = _State(), np.random.default_rng(int(seed))
    s.codec = _circ16(case["size"])
    data = np.zeros(s.codec.message_size, np.uint8)
    data[:case["size"]] = rng.integers(0, 256, case["size"], dtype=np.uint8)
    s.msg = bytearray(data.tobytes())
    ecc = np.frombuffer(bytes(s.codec.encode(s.msg)), np.uint8).copy()
    lost = int(case["size"] * case["lost"])  # a lost stretch of the file, and single damaged bytes
    at = int(rng.integers(0, case["size"] - lost))
    data[at:at + lost] = rng.integers(0, 256, lost, dtype=np.uint8)
    one = rng.integers(0, case["size"], 16)
    data[one] ^= rng.integers(1, 256, 16, dtype=np.uint8)
    one = rng.integers(0, ecc.size, 4)
    ecc[one] ^= rng.integers(1, 256, 4, dtype=np.uint8)
    s.bad_msg, s.bad_par = data.tobytes(), ecc.tobytes()
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "call":
        s = _prepare_call(case, seed)
    elif kind == "circ16":
        s = _prepare_circ16(case, seed)
    elif kind == "mixed":
        s = _prepare_mixed(case, seed)
    else:
        s = _prepare_batch(case, seed)
    s.kind = kind
    return s


# ---- one pass ----------------------------------------------------------------------------------


def _run_host(s, dtype):
    parity = s.codec.encode(s.msg)
    msg, ecc = bytearray(s.bad_msg), bytearray(s.bad_par)
    status = s.codec.repair(msg, ecc)
    return [np.frombuffer(b, dtype) for b in (parity, msg, ecc)] + [int(status)]


def run(state):
    s = state
    if s.kind == "call":
        return _run_host(s, s.dtype)
    if s.kind == "circ16":
        return _run_host(s, np.uint8)
    if s.kind == "mixed":
        s.plan8.encode(s.v_msg[0], s.v_par[0])
        s.plan16.encode(s.v_msg[1], s.v_par[1])
        for i, plan in enumerate(s.plans):
            s.v_fix_msg[i].copy_from(s.v_bad_msg[i])
            s.v_fix_par[i].copy_from(s.v_bad_par[i])
            plan.repair(s.v_fix_msg[i], s.v_fix_par[i], s.v_status[i])
        return [s.par, s.fix_msg, s.fix_par, s.status]
    if s.kind == "rs256_encode":
        s.codec.encode_device(s.k, s.v_msg, s.count, s.v_par)
        return s.par
    if s.kind == "rsi16_encode":
        s.codec.encode_device(s.v_msg, s.count, s.v_par)
        return s.par
    s.v_msg.copy_from(s.v_bad_msg)
    s.v_par.copy_from(s.v_bad_par)
    if s.rs256:
        s.codec.repair_device(s.k, s.v_msg, s.v_par, s.count, s.v_status)
    else:
        s.codec.repair_device(s.v_msg, s.v_par, s.count, s.v_status)
    return [s.msg, s.par, s.status]


# ---- the bytes a pass cannot do without --------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "call":
        n = (case["k"] + case["ecc"]) * (1 if case["field"] == "rs256" else 2)
        return {"bytes": 3 * n + 1, "flops": 0}
    if kind == "circ16":
        c = choose_geometry(case["size"])
        message = (c[0] - c[1]) * c[4] * (c[2] - c[3]) * 2
        ecc = c[3] * (c[0] - c[1]) * c[4] * 2 + c[2] * c[4] * c[1] * 2
        return {"bytes": 3 * (message + ecc), "flops": 0}
    if kind == "mixed":  # mean lengths of the two lists
        rs256 = sum(e + (256 - e) / 2 for e in MIXED_RS256_ECC) / len(MIXED_RS256_ECC)
        rsi16 = 2 * sum(MIXED_RSI16_N) / len(MIXED_RSI16_N)
        return {"bytes": 3 * (case["rs256"] * rs256 + case["rsi16"] * rsi16) + case["rs256"] + case["rsi16"], "flops": 0}
    n = case["k"] + case["ecc"] if kind.startswith("rs256") else 2 * case["n"]
    return {"bytes": case["count"] * (n if kind.endswith("encode") else 2 * n + 1), "flops": 0}


def exact(case, seed):
    """No value: every output is an exact symbol, byte or status code, none is rounded."""
    return None
