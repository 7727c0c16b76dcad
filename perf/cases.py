"""The workloads the library's speed is judged on.

Each case is one call that a prover makes through `zkmetal_amd.MetalMSM`: a
multi-scalar multiplication over BN254 G1, Grumpkin or BN254 G2 with bases and
scalars in device memory, the same with pageable host buffers, MSMs over
prefixes of a resident SRS (alone, as a batch of mixed sizes, on witness-like
scalars) and KZG commitments.  Sizes run from 2^6 points, where launches and
waits are the whole cost, to the 2^22 of the headline benchmark.
"""
import math
import random

import numpy as np

import zkmetal_amd as zk

P = 0x30644e72e131a029b85045b68181585d97816a916871ca8d3c208c16d87cfd47
R = 0x30644e72e131a029b85045b68181585d2833e84879b9709143e1f593f0000001

# name: (coordinate field, group order, generator with coordinates c0 + c1 u,
#        u^2 = -1, half-scalars per scalar, bits of a half-scalar,
#        field multiplies of a mixed and of a full addition, point bytes)
CURVES = {
    "bn254": (P, R, ((1, 0), (2, 0)), 2, 128, 10, 14, 64),
    "grumpkin": (R, P, ((1, 0), (0x2cf135e7506a45d632d270d45f1181294833fc48d823f272c, 0)), 1, 254, 10, 14, 64),
    "g2": (P, R, ((0x1800deef121f1e76426a00665e5c4479674322d4f75edadd46debd5cd992f6ed,
                   0x198e9393920d483a7260bfb731fb5d25f1aa493335a9e71297e485b7aef312c2),
                  (0x12c85ea5db8c6deb4aab71808dcb408fe3d1e7690c43d37b4ce6cc0166fa7daa,
                   0x090689d0585ff075ec9e99ad690c3395bc4b313370b38ef355acdadcd122975b)), 1, 254, 28, 40, 128),
}


def listed():
    return [
        # a verifier's or a small circuit's MSM through the drop-in host call:
        # nothing but launches, waits and the serial tail
        {"name": "host_256", "path": "host", "curve": "bn254", "n": 256},
        # a small commitment whose operands already sit in device memory, one
        # point past a power of two
        {"name": "device_4097", "path": "device", "curve": "bn254", "n": 4097},
        # the per-column commitment of a mid-sized circuit
        {"name": "device_2p16", "path": "device", "curve": "bn254", "n": 1 << 16},
        # the two sizes of the headline metric
        {"name": "device_2p20", "path": "device", "curve": "bn254", "n": 1 << 20},
        {"name": "device_2p22", "path": "device", "curve": "bn254", "n": 1 << 22},
        # the drop-in host call on a circuit of odd size: upload of bases and
        # scalars, table build and MSM
        {"name": "host_400009", "path": "host", "curve": "bn254", "n": 400009},
        # one proving request as a service sees it: witness-like scalars from
        # host memory over a resident SRS
        {"name": "request_150001", "path": "request", "curve": "bn254", "n": 150001, "dist": 1},
        # a proof's commitments in one call over a resident SRS, mixed sizes
        {"name": "batch_64", "path": "batch", "curve": "bn254", "msms": 64, "lo": 12, "hi": 20, "mix": 1, "dist": 0},
        # the witness columns of one proof: mostly zeros and small values
        {"name": "witness_32", "path": "batch", "curve": "bn254", "msms": 32, "lo": 18, "hi": 18, "mix": 1, "dist": 1},
        # KZG commitments to eight polynomials held on the device in Montgomery form
        {"name": "kzg_8", "path": "kzg", "curve": "bn254", "msms": 8, "lo": 16, "hi": 16, "mix": 1},
        # the cycle partner curve of a recursive prover
        {"name": "grumpkin_2p22", "path": "device", "curve": "grumpkin", "n": 1 << 22},
        # Groth16's G2 query
        {"name": "g2_2p20", "path": "device", "curve": "g2", "n": 1 << 20},
    ]


def draw(rng):
    path = rng.choice(["device", "device", "device", "host", "request", "batch", "kzg"])
    if path in ("device", "host"):
        curve = rng.choice(["bn254", "bn254", "grumpkin", "g2"])
        top = 20 if curve == "g2" or path == "host" else 22
        return {"path": path, "curve": curve, "n": int(2 ** rng.uniform(6, top))}
    if path == "request":
        return {"path": path, "curve": "bn254", "n": int(2 ** rng.uniform(10, 20)), "dist": rng.randrange(2)}
    while True:
        lo = rng.uniform(8, 16)
        case = {"path": path, "curve": "bn254", "msms": int(2 ** rng.uniform(1, 6)), "lo": lo,
                "hi": lo + rng.uniform(0, 20 - lo), "mix": rng.randrange(1 << 30)}
        if path == "batch":
            case["dist"] = rng.randrange(2)
        if sum(counts_of(case)) <= 8 << 20:
            return case


def counts_of(case):
    """Points of each MSM of a case."""
    if "n" in case:
        return [case["n"]]
    rng = random.Random(case["mix"])
    return [round(2 ** rng.uniform(case["lo"], case["hi"])) for _ in range(case["msms"])]


def seeds_of(seed):
    """Seeds of the bases and of the scalars."""
    return (2 * seed) % (1 << 64), (2 * seed + 1) % (1 << 64)


def prepare(case, seed):
    base_seed, scalar_seed = seeds_of(seed)
    counts = counts_of(case)
    scalars = zk.gen_scalars(scalar_seed, sum(counts), case.get("dist", 0))
    state = {"case": case, "counts": counts, "engine": zk.MetalMSM()}
    if case["path"] in ("device", "host"):
        points = _points(case["curve"], base_seed, counts[0])
        if case["path"] == "device":
            state["points"], state["scalars"] = points, _on_device(scalars)
        else:
            state["points"] = np.frombuffer(points.download(), dtype=np.uint8)
            state["scalars"] = scalars
        return state
    state["engine"].srs_generate(base_seed, max(counts))
    state["scalars"] = scalars if case["path"] == "request" else _on_device(scalars)
    return state


def _on_device(array):
    buf = zk.DeviceBuffer(array.nbytes)
    buf.upload(array)
    return buf


def _points(curve, seed, n):
    """n affine points k_i G in device memory, in the form the calls take."""
    maker = zk.MetalMSM()
    if curve == "bn254":
        maker.set_window_shift(maker.SHIFT_OFF)
        maker.srs_generate(seed, n)
        points = _on_device(maker.srs_download(n))
    else:
        points = zk.DeviceBuffer(n * CURVES[curve][7])
        make = maker.grumpkin_points_generate if curve == "grumpkin" else maker.g2_points_generate
        make(seed, n, points)
    maker.close()
    return points


def run(state):
    eng, case, counts = state["engine"], state["case"], state["counts"]
    if case["path"] == "device":
        call = {"bn254": eng.msm_batch_device, "grumpkin": eng.grumpkin_msm_batch_device,
                "g2": eng.g2_msm_batch_device}[case["curve"]]
        out = call(state["points"], state["scalars"], counts)
    elif case["path"] == "host":
        call = {"bn254": eng.msm, "grumpkin": eng.grumpkin_msm, "g2": eng.g2_msm}[case["curve"]]
        out = [call(state["points"], state["scalars"])]
    elif case["path"] == "kzg":
        out = eng.kzg_commit(state["scalars"], counts)
    else:
        out = eng.msm_batch_resident(state["scalars"], counts)
    return [np.frombuffer(r, dtype=np.uint8) for r in out]


def work(case):
    """Bytes: every scalar, every base (once, though a batch's MSMs share the
    resident ones) and the results.  Operations: 32-bit limb multiplies and
    adds of Pippenger's method at the window width that needs fewest, 136 limb
    products to a field multiply."""
    _, _, _, halves, span, madd, add, point_bytes = CURVES[case["curve"]]
    counts = counts_of(case)
    muls = 0.0
    for n in counts:
        best = math.inf
        for c in range(2, 25):
            w = math.ceil(span / c)
            # of a hundred witness-like scalars 40 are zero, 30 below 2^16,
            # 10 are 1 or -1 and 20 are full
            digits = n * (0.2 * halves * w + 0.4 * math.ceil(16 / c)) if case.get("dist") else n * halves * w
            best = min(best, madd * digits + 2 * add * w * 2 ** (c - 1))
        muls += best
    nbytes = 32 * sum(counts) + point_bytes * max(counts) + 3 * point_bytes // 2 * len(counts)
    return {"bytes": nbytes, "flops": 2 * 136 * muls}


# ---- the expected results: sum s_i (k_i G) = (sum s_i k_i) G

def _words(seed, index, j):
    """Word j of the seeded stream's elements `index` (splitmix64)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.uint64(0x9e3779b97f4a7c15) * (index * np.uint64(64) + np.uint64(j + 1))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
        return z ^ (z >> np.uint64(31))


def _uniform(seed, index):
    """254-bit candidates, the first below R taken: (len(index), 4) words."""
    out = np.zeros((len(index), 4), dtype=np.uint64)
    todo = np.arange(len(index))
    limbs = [np.uint64((R >> (64 * k)) & (2 ** 64 - 1)) for k in range(4)]
    for attempt in range(16):
        cand = np.stack([_words(seed, index[todo], 4 * attempt + t) for t in range(4)], axis=1)
        cand[:, 3] &= np.uint64((1 << 62) - 1)
        less, equal = np.zeros(len(todo), bool), np.ones(len(todo), bool)
        for k in range(3, -1, -1):
            less |= equal & (cand[:, k] < limbs[k])
            equal &= cand[:, k] == limbs[k]
        out[todo[less]] = cand[less]
        todo = todo[~less]
        if not len(todo):
            return out
    raise ValueError("sixteen rejections in a row")


def _scalars(seed, n, dist):
    index = np.arange(n, dtype=np.uint64)
    if not dist:
        return _uniform(seed, index)
    out = np.zeros((n, 4), dtype=np.uint64)
    cls = _words(seed, index, 60) % np.uint64(100)
    small, unit, full = (cls >= 40) & (cls < 70), (cls >= 70) & (cls < 80), cls >= 80
    out[small, 0] = _words(seed, index[small], 61) & np.uint64(0xffff)
    minus = (_words(seed, index, 62) & np.uint64(1)).astype(bool)
    out[unit & ~minus, 0] = 1
    for k in range(4):
        out[unit & minus, k] = ((R - 1) >> (64 * k)) & (2 ** 64 - 1)
    out[full] = _uniform(seed, index[full])
    return out


def _dot(a, b):
    """sum a_i b_i over 256-bit integers given as 64-bit words, from exact
    double products of their 16-bit digits."""
    total = np.zeros((16, 16), dtype=object)
    for i in range(0, len(a), 1 << 20):
        x = a[i:i + (1 << 20)].view(np.uint16).astype(np.float64)
        y = b[i:i + (1 << 20)].view(np.uint16).astype(np.float64)
        total += (x.T @ y).astype(np.int64).astype(object)
    return sum(int(total[i, j]) << (16 * (i + j)) for i in range(16) for j in range(16))


def _mul(a, b, p):
    return (a[0] * b[0] - a[1] * b[1]) % p, (a[0] * b[1] + a[1] * b[0]) % p


def _add(s, t, p):
    """Sum of two affine points on y^2 = x^3 + b (None: the identity)."""
    if s is None or t is None:
        return s or t
    (x1, y1), (x2, y2) = s, t
    if x1 == x2:
        if ((y1[0] + y2[0]) % p, (y1[1] + y2[1]) % p) == (0, 0):
            return None
        xx = _mul(x1, x1, p)
        num, den = (3 * xx[0], 3 * xx[1]), (2 * y1[0], 2 * y1[1])
    else:
        num, den = (y2[0] - y1[0], y2[1] - y1[1]), (x2[0] - x1[0], x2[1] - x1[1])
    inv = pow(den[0] * den[0] + den[1] * den[1], -1, p)
    m = _mul(num, (den[0] * inv, -den[1] * inv), p)
    mm = _mul(m, m, p)
    x3 = ((mm[0] - x1[0] - x2[0]) % p, (mm[1] - x1[1] - x2[1]) % p)
    y3 = _mul(m, (x1[0] - x3[0], x1[1] - x3[1]), p)
    return x3, ((y3[0] - y1[0]) % p, (y3[1] - y1[1]) % p)


def _result(k, curve):
    """k G as the calls return it: X | Y | 1, Montgomery form, little-endian."""
    p, order, gen = CURVES[curve][:3]
    acc = None
    for bit in bin(k % order)[2:]:
        acc = _add(acc, acc, p)
        if bit == "1":
            acc = _add(acc, gen, p)
    x, y, z = ((1, 0), (1, 0), (0, 0)) if acc is None else (acc[0], acc[1], (1, 0))
    parts = 2 if curve == "g2" else 1
    raw = b"".join((v * 2 ** 256 % p).to_bytes(32, "little") for c in (x, y, z) for v in c[:parts])
    return np.frombuffer(raw, dtype=np.uint8)


def exact(case, seed):
    base_seed, scalar_seed = seeds_of(seed)
    counts = counts_of(case)
    keys = _uniform(base_seed, np.arange(max(counts), dtype=np.uint64))
    scalars = _scalars(scalar_seed, sum(counts), case.get("dist", 0))
    out, at = [], 0
    for n in counts:
        k = _dot(scalars[at:at + n], keys[:n])
        if case["path"] == "kzg":  # coefficients in Montgomery form
            k = k * pow(2 ** 256, -1, R) % R
        out.append(_result(k, case["curve"]))
        at += n
    return out
