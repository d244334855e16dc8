"""Performance cases of the pair-counting framework.

Every case is work that a user has the framework do through its public entry
points: `Engine.count`, `Engine.count_batch`, `Engine.count_prepared` and
`Engine.count_lightcone` on samples that lie on the device, and the whole
`MeasureIABox.measure_xi_w` call from host arrays to the HDF5 file.

A case is a dict of plain values.  `prepare` makes its inputs from a seed on
the GPU, `run` is one pass, `work` the pass's unavoidable bytes and FP64
operations, `exact` the same outputs in plain 64-bit torch arithmetic (one
term per pair, no cells, no bin guesses), where that takes seconds.
"""
import math
import os
import tempfile

import numpy as np
import torch

from measure_ia_amd import MeasureIABox, ReadData, binning
from measure_ia_amd.engine import LightconeArrays, SampleArrays, get_engine
from measure_ia_amd.lightcone import rotated_ellipticity, rp_cut_threshold

# FP64 operations per in-domain pair: separations 3, squared separation 3,
# e+ and ex 14, bins and sums 8 (four more in (r, mu) for r^2 and mu); a
# lightcone pair has two per-axis scales instead.
FLOP = {"rppi": 28, "rmu": 32, "lightcone": 30}
EXACT_PAIRS = 5.0e10     # (shape, position) combinations that exact() goes through at most
CHUNK = 1 << 23          # combinations of one step of exact()

# A wedge of sky and distance like a photometric survey's: RA, DEC (degrees), chi (Mpc).
WEDGE = {"ra_lo": 0.0, "ra_hi": 60.0, "dec_lo": -15.0, "dec_hi": 15.0, "chi_lo": 300.0, "chi_hi": 2000.0}
# Projected correlations on the defaults of a w_gg / w_g+ measurement.
W_BINS = {"mode": "rppi", "r_min": 0.1, "r_max": 20.0, "n_r": 10, "n_2": 20, "pi_max": 60.0}
BOX = {"kind": "box", "L": 205.0, "los": 2, "weights": False, "variance": False, "deterministic": False,
       "clustered": True}
W_BOX, W_WEDGE = {**BOX, **W_BINS}, {**WEDGE, **W_BINS}


def listed():
    return [
        # A small subsample (one mass or colour bin of a small snapshot) on the
        # constructor's default bins, pi_max = L/2, no jackknife: latency.
        dict(BOX, name="box_w_2k", n_pos=2000, n_shape=2000, jk=0, mode="rppi", r_min=0.1, r_max=20.0, n_r=8,
             n_2=20, pi_max=102.5, clustered=False),
        # An ordinary simulation sample with 27 jackknife regions, all galaxies
        # both positions and shapes.
        dict(W_BOX, name="box_w_20k_jk27", n_pos=20000, n_shape=20000, jk=3, clustered=False),
        # The headline measurement: one million clustered galaxies, a fifth of
        # them with shapes.
        dict(W_BOX, name="box_w_1m_jk27", n_pos=1000000, n_shape=200000, jk=3),
        # Multipoles on the same box to large separations, 64 regions.
        dict(BOX, name="box_multipoles_2m_jk64", n_pos=2000000, n_shape=500000, jk=4, mode="rmu", r_min=0.1,
             r_max=60.0, n_r=15, n_2=20, pi_max=0.0),
        # Weighted samples of odd sizes along another line of sight, with the
        # per-bin variance of the single-process layout.
        dict(W_BOX, name="box_w_317k_weighted_var", n_pos=317811, n_shape=75025, jk=3, los=0, weights=True,
             variance=True),
        # A large box to 100 Mpc/h with fine pi bins and 125 regions: the
        # longest single count.
        dict(BOX, name="box_w_3m_r100_jk125", L=500.0, n_pos=3000000, n_shape=750000, jk=5, mode="rppi", r_min=0.1,
             r_max=100.0, n_r=15, n_2=40, pi_max=100.0),
        # A count that has to give the same bits on every run.
        dict(W_BOX, name="box_w_200k_deterministic", n_pos=200000, n_shape=50000, jk=3, deterministic=True),
        # Twelve uneven weighted samples of one box in one call (bins in mass,
        # redshift or colour): the batched count.
        dict(W_BOX, name="batch12_uneven", kind="batch", n_samples=12, n_lo=10000, n_hi=800000, shape_frac=0.3,
             jk=3, weights=True),
        # A lightcone measurement: weighted positions and shapes, 27 patches.
        dict(W_WEDGE, kind="lightcone", name="lightcone_w_1m", n_pos=1000000, n_shape=300000, patches_ra=9,
             patches_dec=3, shapes=True, weights=True, clustered=True, h=1.0, rp_cut=0.0),
        # The random-random count of the lightcone estimators.
        dict(W_WEDGE, kind="lightcone", name="lightcone_rr_4m", n_pos=4000000, n_shape=4000000, patches_ra=9,
             patches_dec=3, shapes=False, weights=False, clustered=False, h=1.0, rp_cut=0.0),
        # A small spectroscopic sample: lightcone multipoles with an r_p cut.
        dict(kind="lightcone", name="lightcone_multipoles_20k", n_pos=20011, n_shape=8009, patches_ra=4,
             patches_dec=2, ra_lo=10.0, ra_hi=40.0, dec_lo=-10.0, dec_hi=10.0, chi_lo=200.0, chi_hi=1400.0,
             mode="rmu", r_min=0.1, r_max=60.0, n_r=15, n_2=20, pi_max=0.0, shapes=True, weights=True,
             clustered=True, h=0.7, rp_cut=0.5),
        # The whole call: host arrays in, prepared sample and count on the
        # device, estimators, 27 realisations and the HDF5 file.
        dict(W_BOX, kind="measure", name="measure_xi_w_300k", n_pos=300000, n_shape=60000, jk=3),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, sizes spread over the logarithm of the listed range."""
    kind = rng.choice(["box", "box", "box", "box", "prepared", "batch", "lightcone", "lightcone", "lightcone",
                       "measure"])
    if kind == "lightcone":
        n_pos = _log_uniform(rng, 3000, 2000000)
        shapes = rng.random() < 0.7
        span = 25.0 + 35.0 * rng.random()
        lo = 200.0 + 200.0 * rng.random()
        c = dict(kind=kind, n_pos=n_pos, n_shape=max(500, int(n_pos * rng.uniform(0.15, 1.0))),
                 patches_ra=rng.choice([0, 3, 5, 9]), patches_dec=rng.choice([2, 3]), ra_lo=5.0, ra_hi=5.0 + span,
                 dec_lo=-0.25 * span, dec_hi=0.25 * span, chi_lo=lo, chi_hi=lo + rng.uniform(900.0, 1700.0),
                 shapes=shapes, weights=rng.random() < 0.6, clustered=rng.random() < 0.6,
                 h=rng.choice([1.0, 0.7]), rp_cut=0.0)
        c.update(_draw_bins(rng, 0.0, n_pos * c["n_shape"] < 2e10))
        if c["mode"] == "rmu":
            c["rp_cut"] = rng.choice([0.0, 0.5, 1.0])
        while _pairs(c) > 5.0e9:
            c["n_pos"] = int(c["n_pos"] * 0.7)
            c["n_shape"] = int(c["n_shape"] * 0.7)
        return c
    L = rng.choice([75.0, 205.0, 205.0, 300.0, 500.0])
    c = dict(BOX, kind=kind, L=L, los=rng.choice([0, 1, 2, 2]), clustered=rng.random() < 0.7)
    if kind == "batch":
        c.update(W_BINS, n_samples=rng.choice([3, 5, 8, 12]), n_lo=_log_uniform(rng, 2000, 20000),
                 n_hi=_log_uniform(rng, 40000, 400000), shape_frac=rng.uniform(0.1, 0.5), jk=rng.choice([2, 3]),
                 weights=rng.random() < 0.6, L=max(L, 205.0))
        return c
    n_pos = _log_uniform(rng, 1000, 1500000)
    c.update(n_pos=n_pos, n_shape=n_pos if rng.random() < 0.25 else max(200, int(n_pos * rng.uniform(0.05, 0.6))),
             jk=rng.choice([0, 2, 3, 3, 4]), weights=rng.random() < 0.4)
    if L < 100.0:  # the same number density as a larger box, so that reach and box stay apart
        c.update(n_pos=min(c["n_pos"], 300001), n_shape=min(c["n_shape"], 100003))
    if kind == "measure":
        c.update(W_BINS, n_pos=min(c["n_pos"], 400009), n_shape=min(c["n_shape"], 100003), jk=rng.choice([2, 3]),
                 pi_max=min(60.0, L / 2.0))
        return c
    c.update(_draw_bins(rng, L, n_pos <= 300000))
    if kind == "box":
        c["variance"] = rng.random() < 0.25
        c["deterministic"] = n_pos <= 500000 and rng.random() < 0.2
    while _pairs(c) > 6.0e10:
        c["n_pos"] = int(c["n_pos"] * 0.7)
        c["n_shape"] = int(c["n_shape"] * 0.7)
    return c


def _draw_bins(rng, L, fine):
    """Binnings in use: projected or (r, mu), 8 to 15 r bins, now and then a fine grid."""
    top = 20.0 if L and L < 150.0 else rng.choice([20.0, 20.0, 30.0, 60.0])
    n_r, n_2 = rng.choice([(8, 20), (10, 20), (15, 20), (12, 30), (40, 40) if fine else (10, 20)])
    if rng.random() < 0.4:
        return dict(mode="rmu", r_min=0.1, r_max=top, n_r=n_r, n_2=n_2, pi_max=0.0)
    pi_max = rng.choice([30.0, 60.0, 60.0, 100.0])
    if L:
        pi_max = min(pi_max, L / 2.0)
    return dict(mode="rppi", r_min=rng.choice([0.1, 0.1, 0.5]), r_max=top, n_r=n_r, n_2=n_2, pi_max=pi_max)


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _positions(g, n, L, clustered):
    """n points of the box: uniform, or three quarters in Gaussian clusters of about 150 (sigma 1)."""
    x = _rand(g, n, 3) * L
    if clustered:
        m = int(0.75 * n)
        centres = _rand(g, max(1, m // 150), 3) * L
        which = torch.randint(0, len(centres), (m,), generator=g, device="cuda")
        x[:m] = centres[which] + _randn(g, m, 3)
        x = torch.remainder(x, L)
        x = torch.where(x >= L, torch.zeros_like(x), x)
        x = x[torch.randperm(n, generator=g, device="cuda")].contiguous()
    return x


def _ellipticities(g, n):
    e12 = 0.22 * _randn(g, n, 2)
    e = torch.linalg.norm(e12, dim=1)
    return e12 * torch.where(e >= 0.95, 0.95 / e, torch.ones_like(e))[:, None]


def _box_sample(g, c, n_pos, n_shape):
    """Positions, a random subset of them as shape sample, axes, |e| and weights, as the counters take them."""
    pos = _positions(g, n_pos, c["L"], c["clustered"])
    n_shape = min(n_shape, n_pos)
    shp = pos if n_shape == n_pos else pos[torch.randperm(n_pos, generator=g, device="cuda")[:n_shape]].contiguous()
    e12 = _ellipticities(g, n_shape)
    theta = 0.5 * torch.atan2(e12[:, 1], e12[:, 0])
    axis = torch.stack([torch.cos(theta), torch.sin(theta)], dim=1)
    w = ws = None
    if c["weights"]:
        w, ws = 0.5 + _rand(g, n_pos), 0.5 + _rand(g, n_shape)
    return SampleArrays(positions=pos, shapes=shp, axis=axis, e=torch.linalg.norm(e12, dim=1), weight=w,
                        weight_shape=ws, boxsize=c["L"], los=c["los"], jk_per_side=c["jk"],
                        jk_sub=c["L"] / c["jk"] if c["jk"] else 0.0)


def _batch_sizes(c):
    """Uneven sample sizes, evenly spaced in the logarithm, the largest neither first nor last."""
    n = c["n_samples"]
    sizes = [int(c["n_lo"] * (c["n_hi"] / c["n_lo"]) ** (i / (n - 1.0))) | 1 for i in range(n)]
    return sizes[n // 2:] + sizes[:n // 2]


def _edges(c):
    r_bins = np.logspace(np.log10(c["r_min"]), np.log10(c["r_max"]), c["n_r"] + 1)
    if c["mode"] == "rppi":
        return r_bins, np.linspace(-c["pi_max"], c["pi_max"], c["n_2"] + 1)
    return r_bins, np.linspace(-1, 1, c["n_2"] + 1)


def _thresholds(c):
    r_bins, second = _edges(c)
    make = binning.rppi_thresholds if c["mode"] == "rppi" else binning.rmu_thresholds
    return make(r_bins, second, c["r_min"], c["r_max"])


def _wedge(g, c, n):
    """n objects of the wedge, uniform in volume, half of them in clusters where the case asks for it."""
    ra = c["ra_lo"] + (c["ra_hi"] - c["ra_lo"]) * _rand(g, n)
    s0, s1 = math.sin(math.radians(c["dec_lo"])), math.sin(math.radians(c["dec_hi"]))
    dec = torch.rad2deg(torch.asin(s0 + (s1 - s0) * _rand(g, n)))
    chi = (c["chi_lo"] ** 3 + (c["chi_hi"] ** 3 - c["chi_lo"] ** 3) * _rand(g, n)) ** (1.0 / 3.0)
    if c["clustered"]:
        m = n // 2
        head = torch.randint(0, max(1, m // 50), (m,), generator=g, device="cuda") + m  # centres: unclustered objects
        head = torch.clamp(head, max=n - 1)
        step = 1.5 * _randn(g, m, 3)
        k = 180.0 / (math.pi * chi[head])
        ra[:m] = ra[head] + step[:, 0] * k / torch.cos(torch.deg2rad(dec[head]))
        dec[:m] = dec[head] + step[:, 1] * k
        chi[:m] = torch.clamp(chi[head] + step[:, 2], c["chi_lo"], c["chi_hi"])
        p = torch.randperm(n, generator=g, device="cuda")
        ra, dec, chi = ra[p], dec[p], chi[p]
    return ra.contiguous(), dec.contiguous(), chi.contiguous()


def _patches(c, ra, dec):
    if not c["patches_ra"]:
        return None
    i = ((ra - c["ra_lo"]) / (c["ra_hi"] - c["ra_lo"]) * c["patches_ra"]).long().clamp(0, c["patches_ra"] - 1)
    j = ((dec - c["dec_lo"]) / (c["dec_hi"] - c["dec_lo"]) * c["patches_dec"]).long().clamp(0, c["patches_dec"] - 1)
    return (i * c["patches_dec"] + j).to(torch.int32)


def _lightcone_sample(g, c):
    n, m = c["n_pos"], c["n_shape"]
    ra, dec, chi = _wedge(g, c, n)
    if not c["shapes"] and m == n:
        sel = slice(None)  # randoms against themselves
    else:
        sel = torch.randint(0, n, (m,), generator=g, device="cuda")
    ra_s, dec_s, chi_s = ra[sel].contiguous(), dec[sel].contiguous(), chi[sel].contiguous()
    c2 = s2 = None
    if c["shapes"]:
        e12 = _ellipticities(g, m).cpu().numpy()
        c2, s2 = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in rotated_ellipticity(e12[:, 0], e12[:, 1]))
    return LightconeArrays(ra=ra, dec=dec, chi=chi, cos_dec=torch.cos(dec / 180 * math.pi), ra_s=ra_s, dec_s=dec_s,
                           chi_s=chi_s, weight=0.5 + _rand(g, n) if c["weights"] else None,
                           weight_shape=0.5 + _rand(g, m) if c["weights"] else None, c2=c2, s2=s2,
                           patch=_patches(c, ra, dec), patch_s=_patches(c, ra_s, dec_s),
                           n_patches=c["patches_ra"] * c["patches_dec"], proj_scale=c["h"],
                           rp2_cut=rp_cut_threshold(c["rp_cut"]))


def _measure_data(g, c):
    """The data dict a user hands to MeasureIABox."""
    s = _box_sample(g, c, c["n_pos"], c["n_shape"])
    e = s.e.cpu().numpy()
    data = {"Position": s.positions.cpu().numpy(), "Position_shape_sample": s.shapes.cpu().numpy(),
            "Axis_Direction": s.axis.cpu().numpy(), "LOS": c["los"], "q": np.sqrt((1.0 - e) / (1.0 + e))}
    if c["weights"]:
        data["weight"] = s.weight.cpu().numpy()
        data["weight_shape_sample"] = s.weight_shape.cpu().numpy()
    return data


def prepare(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "measure":
        return {"case": c, "data": _measure_data(g, c), "folder": tempfile.TemporaryDirectory()}
    st = {"case": c, "engine": get_engine(0), "bins": _thresholds(c)}
    if c["kind"] == "lightcone":
        st["sample"] = _lightcone_sample(g, c)
    elif c["kind"] == "batch":
        st["samples"] = [_box_sample(g, c, n, max(1, int(c["shape_frac"] * n))) for n in _batch_sizes(c)]
    else:
        st["sample"] = _box_sample(g, c, c["n_pos"], c["n_shape"])
        st["tuning"] = {"deterministic": 1} if c["deterministic"] else None
    if c["kind"] == "prepared":
        # a program that counts several binnings keeps the sorted sample
        st["handle"] = st["engine"].prepare(st["sample"], st["bins"])
    return st


# ---------------------------------------------------------------------------
# one pass


def _outputs(r):
    out = {"npairs": r.npairs, "dd": r.dd, "splus": r.splus, "scross": r.scross, "variance": r.variance,
           "region_stats": r.region_stats}
    return {k: v for k, v in out.items() if v is not None}


def run(state):
    c = state["case"]
    if c["kind"] == "measure":
        name = os.path.join(state["folder"].name, "out.hdf5")
        if os.path.exists(name):
            os.remove(name)
        box = MeasureIABox(dict(state["data"]), name, None, 99, [c["r_min"], c["r_max"]], c["n_r"], c["n_2"],
                           c["pi_max"], boxsize=c["L"], verbose=False)
        box.measure_xi_w("All", "both", num_jk=c["jk"] ** 3)
        got = ReadData(None, "out", 99, data_path=state["folder"].name)
        got.read_MeasureIA_output("All", c["jk"] ** 3)
        return {k: np.asarray(getattr(got, k)) for k in ("rp", "w_gg", "w_gp", "cov_w_gg", "cov_w_gp", "errors_w_gg",
                                                         "errors_w_gp")}
    eng, th = state["engine"], state["bins"]
    if c["kind"] == "lightcone":
        return _outputs(eng.count_lightcone(state["sample"], th))
    if c["kind"] == "batch":
        return [_outputs(r) for r in eng.count_batch(state["samples"], th, variance=c["variance"])]
    if c["kind"] == "prepared":
        return _outputs(eng.count_prepared([state["handle"]], th, variance=c["variance"])[0])
    return _outputs(eng.count(state["sample"], th, variance=c["variance"], tuning=state["tuning"]))


# ---------------------------------------------------------------------------
# work


def _domain(c):
    if c["mode"] == "rppi":
        return math.pi * (c["r_max"] ** 2 - c["r_min"] ** 2) * 2.0 * c["pi_max"]
    return 4.0 / 3.0 * math.pi * (c["r_max"] ** 3 - c["r_min"] ** 3)


def _pairs(c, n_pos=None, n_shape=None):
    """In-domain pairs at the mean density."""
    n_pos, n_shape = n_pos or c["n_pos"], n_shape or c["n_shape"]
    if c["kind"] == "lightcone":
        sky = math.radians(c["ra_hi"] - c["ra_lo"]) * (math.sin(math.radians(c["dec_hi"]))
                                                       - math.sin(math.radians(c["dec_lo"])))
        volume = sky * (c["chi_hi"] ** 3 - c["chi_lo"] ** 3) / 3.0
        scale = c["h"] ** 2 if c["mode"] == "rppi" else 1.0
        return n_pos * n_shape * min(1.0, _domain(c) / scale / volume)
    return n_pos * n_shape * min(1.0, _domain(c) / c["L"] ** 3)


def work(case):
    """Each input read once, each output written once; the in-domain pairs' arithmetic."""
    c = case
    bins = c["n_r"] * c["n_2"]
    if c["kind"] == "lightcone":
        per_pos = 32 + (8 if c["weights"] else 0) + (4 if c["patches_ra"] else 0)
        per_shp = 24 + (16 if c["shapes"] else 0) + (8 if c["weights"] else 0) + (4 if c["patches_ra"] else 0)
        rows = 1 + c["patches_ra"] * c["patches_dec"]
        out = 8 * bins * rows * (4 if c["shapes"] else 2)
        return {"bytes": c["n_pos"] * per_pos + c["n_shape"] * per_shp + out, "flops": FLOP["lightcone"] * _pairs(c)}
    rows = 1 + c["jk"] ** 3
    out = 8 * bins * (3 * rows + 1 + (1 if c["variance"] else 0)) + 32 * (rows - 1)
    per_pos, per_shp = (32, 56) if c["weights"] else (24, 48)
    if c["kind"] == "batch":
        sizes = _batch_sizes(c)
        return {"bytes": sum(n * (per_pos + c["shape_frac"] * per_shp) + out for n in sizes),
                "flops": sum(FLOP[c["mode"]] * _pairs(c, n, c["shape_frac"] * n) for n in sizes)}
    if c["kind"] == "measure":
        out = 8 * (3 * c["n_r"] + 2 * c["n_r"] ** 2 + 2 * c["n_r"])
    return {"bytes": c["n_pos"] * per_pos + c["n_shape"] * per_shp + out, "flops": FLOP[c["mode"]] * _pairs(c)}


# ---------------------------------------------------------------------------
# the same in 64 bits, pair by pair


def _index(c, r, second):
    """The bin of every pair, from the logarithm of r and the linear second coordinate."""
    step = (math.log10(c["r_max"]) - math.log10(c["r_min"])) / c["n_r"]
    i = torch.floor(torch.log10(r) / step - math.log10(c["r_min"]) / step).long().clamp(max=c["n_r"] - 1)
    lo, width = (-c["pi_max"], 2.0 * c["pi_max"] / c["n_2"]) if c["mode"] == "rppi" else (-1.0, 2.0 / c["n_2"])
    j = torch.floor(second / width - lo / width).long()
    j = torch.where(j < 0, j + c["n_2"], j).clamp(max=c["n_2"] - 1)
    return i * c["n_2"] + j


class _Sums:
    """Sums by key, in copies that consecutive terms take in turn (few terms then wait for the same address)."""

    def __init__(self, size):
        self.size, self.copies = size, max(1, min(4096, (1 << 25) // size))
        self.sums = torch.zeros(self.copies * size, device="cuda", dtype=torch.float64)

    def places(self, key):
        return torch.arange(len(key), device="cuda") % self.copies * self.size + key

    def add(self, places, terms):
        self.sums.index_add_(0, places, terms)

    def total(self):
        return self.sums.reshape(self.copies, self.size).sum(0)


def _tally(sums, K, rows, n_r, n_2):
    """Row 0: all pairs; row 1 + k: the pairs of which either side is in region k."""
    t = sums.total().reshape(K, K, n_r * n_2)
    total = t.sum((0, 1))
    if rows == 1:
        return total.reshape(1, n_r, n_2)
    both = t.sum(1) + t.sum(0) - torch.diagonal(t).transpose(0, 1)
    return torch.cat([total[None], both]).reshape(rows, n_r, n_2)


def _regions(x, jk, L):
    if not jk:
        return torch.zeros(len(x), dtype=torch.long, device="cuda")
    sub = L / jk
    k = torch.floor(x / sub).clamp(0, jk - 1)
    inside = ((x > k * sub) & (x < (k + 1) * sub)).all(1)
    k = k.long()
    return torch.where(inside, (k[:, 0] * jk + k[:, 1]) * jk + k[:, 2], torch.zeros_like(k[:, 0]))


def _box_exact(c, s):
    L, half, los = c["L"], c["L"] / 2.0, c["los"]
    a, b = [k for k in range(3) if k != los]
    n_pos, n_shape, jk = len(s.positions), len(s.shapes), c["jk"]
    if n_pos * n_shape * min(1.0, (2.0 * c["r_max"] + 0.02 * L) / L) > EXACT_PAIRS:
        return None
    op, os_ = torch.argsort(s.positions[:, a]), torch.argsort(s.shapes[:, a])
    pos, shp, axis, e = s.positions[op], s.shapes[os_], s.axis[os_], s.e[os_]
    w = torch.ones(n_pos, device="cuda", dtype=torch.float64) if s.weight is None else s.weight[op]
    ws = torch.ones(n_shape, device="cuda", dtype=torch.float64) if s.weight_shape is None else s.weight_shape[os_]
    rp_, rs_ = _regions(pos, jk, L), _regions(shp, jk, L)
    K, B = max(1, jk ** 3), c["n_r"] * c["n_2"]
    keys = pos[:, a].contiguous()
    dd, sp, sx, var = _Sums(K * K * B), _Sums(K * K * B), _Sums(B), _Sums(B)
    at = 0
    while at < n_shape:
        end = min(n_shape, at + 256)
        lo, hi = float(shp[at, a]) - c["r_max"] * 1.000001, float(shp[end - 1, a]) + c["r_max"] * 1.000001
        parts = [(0, n_pos)]
        if hi - lo < L:
            cut = torch.searchsorted(keys, torch.tensor([lo, hi, lo + L, hi - L], device="cuda",
                                                        dtype=torch.float64)).tolist()
            parts = [(cut[0], cut[1])] + ([(cut[2], n_pos)] if lo < 0 else []) + ([(0, cut[3])] if hi > L else [])
        for p0, p1 in parts:
            step = max(1, CHUNK // max(1, end - at))
            for q0 in range(p0, p1, step):
                q1 = min(p1, q0 + step)
                d = []
                for k in range(3):
                    x = shp[at:end, k, None] - pos[None, q0:q1, k]
                    x = torch.where(x > half, x - L, x)
                    d.append(torch.where(x < -half, x + L, x))
                r = torch.sqrt(d[a] * d[a] + d[b] * d[b])
                if c["mode"] == "rppi":
                    sep, keep = r, (d[los] >= -c["pi_max"]) & (d[los] < c["pi_max"])
                else:
                    sep, keep = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]), r > 0
                i, j = torch.nonzero(keep & (sep >= c["r_min"]) & (sep < c["r_max"]), as_tuple=True)
                dx, dy, dl, r, sep = d[a][i, j], d[b][i, j], d[los][i, j], r[i, j], sep[i, j]
                i, j = i + at, j + q0
                bins = _index(c, sep, dl if c["mode"] == "rppi" else dl / sep)
                dot = (dx / r) * axis[i, 0]
                dot = dot + (dy / r) * axis[i, 1]
                phi = torch.arccos(dot)
                ww = w[j] * ws[i]
                ep, ex = (torch.nan_to_num(e[i] * f(2.0 * phi), nan=0.0) * ww for f in (torch.cos, torch.sin))
                places = dd.places((rs_[i] * K + rp_[j]) * B + bins)
                dd.add(places, ww)
                sp.add(places, ep)
                places = sx.places(bins)
                sx.add(places, ex)
                if c["variance"]:
                    var.add(places, ep * ep)
        at = end
    rows = 1 + jk ** 3
    shape = (c["n_r"], c["n_2"])
    out = {"npairs": None, "dd": _tally(dd, K, rows, *shape), "splus": _tally(sp, K, rows, *shape),
           "scross": sx.total().reshape(shape)}
    if c["variance"]:
        out["variance"] = var.total().reshape(shape)
    if jk:
        st = torch.zeros(K, 4, device="cuda", dtype=torch.float64)
        st[:, 0] = torch.bincount(rp_, minlength=K)
        st[:, 1] = torch.bincount(rs_, minlength=K)
        st[:, 2].index_add_(0, rs_, ws)
        st[:, 3].index_add_(0, rs_, ws * (1 - e * e / 2.0))
        out["region_stats"] = st
    return {k: v if v is None else v.cpu().numpy() for k, v in out.items()}


def _lightcone_exact(c, s):
    n_pos, n_shape, K, B = c["n_pos"], c["n_shape"], max(1, s.n_patches), c["n_r"] * c["n_2"]
    reach = (c["pi_max"] if c["mode"] == "rppi" else c["r_max"]) * 1.000001
    if n_pos * n_shape * min(1.0, 3.0 * reach / (c["chi_hi"] - c["chi_lo"])) > EXACT_PAIRS:
        return None
    op, os_ = torch.argsort(s.chi), torch.argsort(s.chi_s)
    ra, dec, chi, cosd = s.ra[op], s.dec[op], s.chi[op].contiguous(), s.cos_dec[op]
    ra_s, dec_s, chi_s = s.ra_s[os_], s.dec_s[os_], s.chi_s[os_]
    one = {"device": "cuda", "dtype": torch.float64}
    w = torch.ones(n_pos, **one) if s.weight is None else s.weight[op]
    ws = torch.ones(n_shape, **one) if s.weight_shape is None else s.weight_shape[os_]
    pp = s.patch[op].long() if s.patch is not None else torch.zeros(n_pos, dtype=torch.long, device="cuda")
    ps = s.patch_s[os_].long() if s.patch_s is not None else torch.zeros(n_shape, dtype=torch.long, device="cuda")
    names = ("dd", "splus", "scross") if c["shapes"] else ("dd",)
    sums = {k: _Sums(K * K * B) for k in names}
    if c["shapes"]:
        c2, s2 = s.c2[os_], s.s2[os_]
    at = 0
    while at < n_shape:
        end = min(n_shape, at + 256)
        p0, p1 = torch.searchsorted(chi, torch.stack([chi_s[at] - reach, chi_s[end - 1] + reach])).tolist()
        step = max(1, CHUNK // (end - at))
        for q0 in range(p0, p1, step):
            q1 = min(p1, q0 + step)
            pi = chi_s[at:end, None] - chi[None, q0:q1]
            dx = ((ra_s[at:end, None] - ra[None, q0:q1]) / 180 * math.pi) * chi[None, q0:q1] * cosd[None, q0:q1]
            dy = ((dec_s[at:end, None] - dec[None, q0:q1]) / 180 * math.pi) * chi[None, q0:q1]
            hx, hy = dx * c["h"], dy * c["h"]
            r = torch.sqrt(hx * hx + hy * hy)
            if c["mode"] == "rppi":
                sep, keep = r, (pi >= -c["pi_max"]) & (pi < c["pi_max"])
            else:
                sep, keep = torch.sqrt(dx * dx + dy * dy + pi * pi), r > c["rp_cut"]
            i, j = torch.nonzero(keep & (sep >= c["r_min"]) & (sep < c["r_max"]), as_tuple=True)
            dx, dy, pi, sep = dx[i, j], dy[i, j], pi[i, j], sep[i, j]
            i, j = i + at, j + q0
            bins = _index(c, sep, pi if c["mode"] == "rppi" else pi / sep)
            places = sums["dd"].places((ps[i] * K + pp[j]) * B + bins)
            ww = w[j] * ws[i]
            sums["dd"].add(places, ww)
            if c["shapes"]:
                rr = dx * dx + dy * dy
                cos2, sin2 = (dx * dx - dy * dy) / rr, 2.0 * dx * dy / rr
                sums["splus"].add(places, ww * (c2[i] * cos2 + s2[i] * sin2))
                sums["scross"].add(places, ww * (s2[i] * cos2 - c2[i] * sin2))
        at = end
    rows = 1 + s.n_patches
    out = {k: _tally(v, K, rows, c["n_r"], c["n_2"]).cpu().numpy() for k, v in sums.items()}
    return dict(out, npairs=None)


def _measure_exact(c, data):
    """w_gg and w_g+ of the whole call, by the estimators' formulas."""
    cuda = {k: torch.from_numpy(v).cuda() for k, v in data.items() if isinstance(v, np.ndarray)}
    axis = cuda["Axis_Direction"]
    axis = axis / torch.sqrt(axis[:, 0] ** 2 + axis[:, 1] ** 2)[:, None]
    e = (1 - cuda["q"] ** 2) / (1 + cuda["q"] ** 2)
    s = SampleArrays(positions=cuda["Position"], shapes=cuda["Position_shape_sample"], axis=axis, e=e,
                     weight=cuda.get("weight"), weight_shape=cuda.get("weight_shape_sample"))
    got = _box_exact(dict(c, jk=0), s)
    if got is None:
        return None
    ws = s.weight_shape.cpu().numpy() if s.weight_shape is not None else np.ones(len(e))
    en = e.cpu().numpy()
    R = float(np.sum(ws * (1 - en ** 2 / 2.0)) / np.sum(ws))
    r_bins, pi_bins = _edges(c)
    dpi = np.diff(pi_bins)
    rr = (len(s.positions) * len(s.shapes) * math.pi * np.diff(r_bins ** 2)[:, None] * dpi[None, :]) / c["L"] ** 3
    none = {k: None for k in ("cov_w_gg", "cov_w_gp", "errors_w_gg", "errors_w_gp")}
    return dict(none, rp=(r_bins[1:] + r_bins[:-1]) / 2.0, w_gg=((got["dd"][0] / rr - 1.0) * dpi).sum(1),
                w_gp=(got["splus"][0] / (2.0 * R) / rr * dpi).sum(1))


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "measure":
        return _measure_exact(c, _measure_data(g, c))
    if c["kind"] == "lightcone":
        return _lightcone_exact(c, _lightcone_sample(g, c))
    if c["kind"] == "batch":
        sizes = _batch_sizes(c)
        near = min(1.0, (2.0 * c["r_max"] + 0.02 * c["L"]) / c["L"])
        if sum(c["shape_frac"] * n * n for n in sizes) * near > EXACT_PAIRS:
            return None
        return [_box_exact(c, _box_sample(g, c, n, max(1, int(c["shape_frac"] * n)))) for n in sizes]
    return _box_exact(c, _box_sample(g, c, c["n_pos"], c["n_shape"]))
