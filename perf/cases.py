"""Timed cases of the GetHI density-to-sky framework, through its public Python entry points.

A case is a dict of plain values; its "kind" names the work:

  mock       one GetHI run into its temperature maps (what the `gethi` program does per parameter file)
  ensemble   several unlike mocks replayed as one graph (crime_amd.Batch)
  training   one training mock of the C_l emulator: a deterministic run and the spectra of its channel pairs
  power      the Gaussian field of a run and its shell-averaged P(k)
  spectra    all cross-frequency C_l of resident maps (map2alm and the pair spectra)
  sky        a mock seen by an instrument: run, beam, noise, mask (map2alm and alm2map)
  sources    a mock with its point-source maps
  predict    binned C_l from the trained emulator's network
  train      a stretch of the network's training from its initial weights

listed() holds the sizes of crime_amd/configs.py, of the emulator and of the small end of each range;
draw() spreads over the same ranges.  Outputs that live on the device come back as views of the
framework's own buffers.
"""
import ctypes
import math
import tempfile

import numpy as np
import torch

import crime_amd
import crime_amd.configs as cf
import crime_amd.emulator as em

NU_21 = 1420.40575177
DEV = "cuda"

# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
ENSEMBLE_KINDS = {"a": 0, "b": 32, "c": 64}   # first member of each kind in configs.ensemble_member


def _mock(name, **kw):
    c = dict(kind="mock", n_grid=256, n_side=128, n_nu=64, nu_lo=700.0, nu_hi=800.0, l_box=-1.0, n_subcell=0,
             fp64=False, bias="reference", velocity="stencil", deterministic=False, tuned=False)
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest run a user makes (a test of a parameter file): launches and synchronisations count
        _mock("mock_64_fp64", n_grid=64, n_side=32, n_nu=16, n_subcell=2, fp64=True),
        # the production mock (configs.production_1024), with the schedule its autotuner saved
        _mock("mock_1024", n_grid=1024, n_side=512, n_nu=200, nu_lo=400.0, l_box=8300.0, bias="linear", tuned=True),
        # the options of configs.largest_2048 (spectral velocities, 4^3 samples a cell) on a ragged grid
        _mock("mock_384_spectral", n_grid=384, n_side=256, n_nu=100, nu_lo=400.0, l_box=8300.0, n_subcell=4,
              velocity="spectral"),
        # two members of each kind of configs.ensemble_member in one graph
        dict(name="ensemble_6", kind="ensemble", members="aabbcc", streams=4),
        # one realisation of the emulator's training set (emulator.simulate)
        dict(name="training_mock", kind="training", n_grid=256, n_side=256, n_nu=64),
        # the P(k) of a realisation, the check every new parameter file gets
        dict(name="power_512", kind="power", n_grid=512, fp64=False, l_box=4000.0),
        # the C_l of the production mock's 200 channels, left on the device
        dict(name="spectra_512x200", kind="spectra", n_side=512, lmax=1535, n_maps=200),
        # configs.small_fp64_256 through the hand-off stages: a 15 m dish, thermal noise, a sky cut
        dict(name="sky_256_fp64", kind="sky", n_grid=256, n_side=128, n_nu=64, l_box=4900.0, n_subcell=2, fp64=True),
        # a low-redshift mock with do_psources
        dict(name="sources_256", kind="sources", n_grid=256, n_side=128, n_nu=32, nu_lo=1050.0, nu_hi=1300.0),
        # one step of a parameter chain: the 256 spectra of one cosmology
        dict(name="predict_1", kind="predict", cosmologies=1, channels=8),
        # a batch of cosmologies, as the emulator is benchmarked
        dict(name="predict_4096", kind="predict", cosmologies=4096, channels=8),
        # training at the emulator's own batch size
        dict(name="train_4096", kind="train", rows=131072, batch=4096, steps=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mock64", "mock32", "spectral", "ensemble", "training", "power", "spectra", "sky", "sources",
                       "predict", "train"])
    if kind == "mock64":
        return _mock(None, n_grid=rng.choice([32, 48, 64, 96, 128, 192, 256]), n_side=_log_int(rng, 16, 128),
                     n_nu=rng.randint(8, 64), n_subcell=rng.choice([0, 1, 2, 3]), fp64=True,
                     l_box=round(rng.uniform(3000.0, 5000.0), 1))
    if kind == "mock32":
        return _mock(None, n_grid=rng.choice([128, 192, 256, 384, 512, 768]), n_side=_log_int(rng, 64, 512),
                     n_nu=rng.randint(32, 200), nu_lo=400.0, bias=rng.choice(["reference", "linear", "const"]),
                     l_box=round(rng.uniform(6000.0, 8300.0), 1), deterministic=rng.random() < 0.3,
                     tuned=rng.random() < 0.5)
    if kind == "spectral":
        return _mock(None, n_grid=rng.choice([96, 128, 192, 256, 384]), n_side=_log_int(rng, 32, 256),
                     n_nu=rng.randint(16, 100), nu_lo=400.0, l_box=round(rng.uniform(6000.0, 8300.0), 1),
                     n_subcell=rng.choice([0, 2, 3, 4]), velocity="spectral")
    if kind == "ensemble":
        return dict(kind="ensemble", members="".join(rng.choice("abc") for _ in range(rng.randint(2, 8))),
                    streams=rng.randint(1, 6))
    if kind == "training":
        return dict(kind="training", n_grid=rng.choice([64, 96, 128, 192, 256]), n_side=_log_int(rng, 32, 256),
                    n_nu=rng.randint(20, 64))
    if kind == "power":
        return dict(kind="power", n_grid=rng.choice([64, 96, 128, 192, 256, 384, 512]), fp64=rng.random() < 0.4,
                    l_box=round(rng.uniform(1000.0, 8000.0), 1))
    if kind == "spectra":
        n_side = _log_int(rng, 16, 512)
        top = 200 if n_side >= 256 else 256
        return dict(kind="spectra", n_side=n_side, lmax=(2 if rng.random() < 0.3 else 3) * n_side - 1,
                    n_maps=_log_int(rng, 1, top))
    if kind == "sky":
        return dict(kind="sky", n_grid=rng.choice([64, 96, 128, 192, 256]), n_side=_log_int(rng, 24, 160),
                    n_nu=rng.randint(5, 64), l_box=round(rng.uniform(3000.0, 5000.0), 1),
                    n_subcell=rng.choice([0, 1, 2]), fp64=rng.random() < 0.5)
    if kind == "sources":
        return dict(kind="sources", n_grid=rng.choice([96, 128, 192, 256]), n_side=_log_int(rng, 32, 256),
                    n_nu=rng.randint(8, 48), nu_lo=round(rng.uniform(1050.0, 1150.0), 1), nu_hi=1300.0)
    if kind == "predict":
        return dict(kind="predict", cosmologies=_log_int(rng, 1, 4096), channels=rng.randint(1, 8))
    return dict(kind="train", rows=_log_int(rng, 20000, 131072), batch=64 * _log_int(rng, 4, 128),
                steps=rng.randint(30, 100))


# ---------------------------------------------------------------------------------------------
# what a user's program has in hand
# ---------------------------------------------------------------------------------------------
class _Device:
    """Device memory of the framework as an array: holds its owner, so that a tensor made of it stays valid."""

    def __init__(self, ptr, shape, fp64, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f8" if fp64 else "<f4",
                                             data=(int(ptr), False), version=2, strides=None)


def _view(ptr, shape, fp64, owner):
    return torch.as_tensor(_Device(ptr, shape, fp64, owner), device=DEV)


def _maps(gh):
    return _view(gh.device_maps()[0], (gh.n_nu, gh.npix), gh.precision == crime_amd.FP64, gh)


def _cosmology(seed):
    rng = np.random.default_rng(seed)
    return dict(omega_m=float(rng.uniform(0.27, 0.33)), sigma_8=float(rng.uniform(0.75, 0.85)))


def _params(case, seed):
    """The parameter file of a case, written and read back as a user's run does."""
    g = dict(n_subcell=0, fp64=False, bias="reference", velocity="stencil", deterministic=False, l_box=-1.0,
             nu_lo=700.0, nu_hi=800.0)
    g.update(case)
    extra = {}
    if g["deterministic"]:
        extra["deterministic"] = 1
    with tempfile.TemporaryDirectory() as tmp:
        bias = {"reference": {}, "const": dict(bias_b0=1.0), "linear": dict(bias_b0=0.7, bias_b1=0.3)}[g["bias"]]
        ini = cf.make(tmp, "case", n_grid=g["n_grid"], n_side=g["n_side"], n_nu=g["n_nu"], nu_lo=g["nu_lo"],
                      nu_hi=g["nu_hi"], l_box=g["l_box"], seed=int(seed) % (1 << 31), bias_model=g["bias"],
                      n_subcell=g["n_subcell"], precision="double" if g["fp64"] else "single",
                      velocity_mode=g["velocity"], extra=extra or None, **bias, **_cosmology(seed))
        return crime_amd.Params(ini)


def _mock_case(case):
    """The GetHI parameters of the kinds that hold one handle."""
    c = dict(case)
    if case["kind"] == "training":
        c.update(bias="const", deterministic=True)
    if case["kind"] == "power":
        c.update(n_side=8, n_nu=4)
    if case["kind"] == "sky":
        c.update(bias="const")
    return c


def _member_params(case, seed):
    pars = []
    with tempfile.TemporaryDirectory() as tmp:
        for i, k in enumerate(case["members"]):
            first = ENSEMBLE_KINDS[k]
            pars.append(crime_amd.Params(cf.ensemble_member(tmp, first + i % 32, seed=(int(seed) + i) % (1 << 31))))
    return pars


def _spec(case):
    if case["kind"] == "training":
        n = case["n_nu"]
        return em.MockSpec(n_grid=case["n_grid"], n_side=case["n_side"], n_nu=n,
                           channels=tuple(int(v) for v in np.linspace(0, n - 2, 8)))
    return em.MockSpec(channels=(0, 9, 18, 27, 36, 45, 54, 62)[:case["channels"]])


def _network(seed, spec, ncos):
    """Raw inputs of ncos cosmologies, and the scaling of a trained emulator over them."""
    x = em.features(em.latin_hypercube(ncos, seed), spec)
    enc = em.encode(em.features(em.latin_hypercube(64, 1), em.MockSpec()), (spec.nu_hi - spec.nu_lo) / spec.n_nu)
    xm, xs = enc.mean(axis=0), enc.std(axis=0)
    return x, dict(x_mean=xm, x_std=xs, y_mean=7.0, y_std=1.5, scale=2e-7, dnu=(spec.nu_hi - spec.nu_lo) / spec.n_nu)


def _training_set(case, seed):
    """Standardised inputs, smooth targets and chi^2 weights of a training set of case["rows"] spectra."""
    rng = np.random.default_rng(seed)
    spec = em.MockSpec()
    x = em.features(em.latin_hypercube(-(-case["rows"] // 256), seed), spec)[: case["rows"]]
    x = em.encode(x, (spec.nu_hi - spec.nu_lo) / spec.n_nu)
    xs = x.std(axis=0)
    xs[xs == 0] = 1.0
    x = ((x - x.mean(axis=0)) / xs).astype(np.float32)
    a = rng.normal(size=8) / math.sqrt(8.0)
    t = np.sin(1.5 * (x @ a)) + 0.4 * x[:, 7] - 0.6 * x[:, 6] + 0.02 * rng.normal(size=len(x))
    w = np.exp(0.7 * rng.normal(size=len(x)))
    return x, t.astype(np.float32), (w / w.mean()).astype(np.float32), em.init_params(seed)


def _sky(case, seed):
    """Beam FWHM and noise per channel of a single-dish survey, and its mask (a band around the equator off)."""
    edges = np.linspace(700.0, 800.0, case["n_nu"] + 1)
    fwhm, sig2 = crime_amd.jt_instrument(edges[:-1], edges[1:], case["n_side"], dish_diameter=15.0, tsys=5e4,
                                         time_total=1000.0, n_dish=200, fsky=0.8)
    npix = 12 * case["n_side"] ** 2
    mask = np.ones(npix, np.uint8)
    mask[int(0.4 * npix): int(0.5 * npix)] = 0
    mask[np.random.default_rng(seed).integers(0, npix, npix // 50)] = 0
    return fwhm, sig2, mask


def _sky_maps(case, seed):
    """Brightness maps of correlated lognormal channels, as the map stage leaves them."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    npix = 12 * case["n_side"] ** 2
    maps = torch.empty((case["n_maps"], npix), dtype=torch.float32, device=DEV)
    prev = torch.randn(npix, generator=g, device=DEV)
    for c in range(case["n_maps"]):
        prev = 0.8 * prev + 0.6 * torch.randn(npix, generator=g, device=DEV)
        maps[c] = 0.1 * torch.exp(0.5 * prev)
    return maps


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, seed=int(seed))
    if kind == "ensemble":
        st["ghs"] = [crime_amd.GetHI(p) for p in _member_params(case, seed)]
        st["batch"] = crime_amd.Batch(st["ghs"], n_streams=case["streams"])
    elif kind == "spectra":
        st["maps"] = _sky_maps(case, seed)
        st["sht"] = crime_amd.Sht(case["n_side"], case["lmax"], max_maps=case["n_maps"])
        torch.cuda.synchronize()
    elif kind == "predict":
        mlp = em.Mlp(max_batch=65536)
        mlp.set_params(em.init_params(int(seed)))
        x, scaling = _network(int(seed), _spec(case), case["cosmologies"])
        st["x"] = x
        st["emu"] = em.Emulator(mlp, **scaling)
    elif kind == "train":
        x, t, w, p = _training_set(case, int(seed))
        st["mlp"] = em.Mlp(max_batch=max(case["batch"], 65536))
        st["mlp"].set_data(x, t, w)
        st.update(p=p, steps=case["steps"], batch=case["batch"])
    else:
        gh = crime_amd.GetHI(_params(_mock_case(case), seed))
        st["gh"] = gh
        if case.get("tuned"):
            gh.set_schedule([3, 1, 1, 1])
        if kind == "training":
            spec = _spec(case)
            st["sht"] = crime_amd.Sht(spec.n_side, spec.lmax, max_maps=spec.n_nu)
            st["pairs"] = spec.pairs
        if kind == "sky":
            st["sht"] = crime_amd.Sht(case["n_side"], max_maps=case["n_nu"])
            st["fwhm"], st["sig2"], st["mask"] = _sky(case, seed)
    return st


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "mock":
        s = st["gh"].run()
        return {"maps": _maps(st["gh"]), "sigma2": s["sigma2_gauss"]}
    if kind == "ensemble":
        st["batch"].run()
        return [_maps(gh) for gh in st["ghs"]]
    if kind == "training":
        gh = st["gh"]
        gh.set_seed(st["seed"])
        gh.run()
        return {"cls": st["sht"].cls_of(gh, pairs=st["pairs"]), "maps": _maps(gh)}
    if kind == "power":
        s = st["gh"].create_d_and_vr_fields()
        k, pk, n = st["gh"].power_spectrum()
        return {"k": k, "pk": pk, "n": n, "sigma2": s["sigma2_gauss"]}
    if kind == "spectra":
        n, _ = st["maps"].shape
        ptr, _ = st["sht"].anafast_device(st["maps"].data_ptr(), n, False, cross=True, to_host=False)
        return {"cls": _view(ptr, (n, n, st["sht"].lmax + 1), True, st["sht"])}
    if kind == "sky":
        gh = st["gh"]
        gh.run()
        st["sht"].instrument_of(gh, fwhm_arcmin=st["fwhm"], sigma2=st["sig2"], seed=st["seed"], mask=st["mask"])
        return {"maps": _maps(gh)}
    if kind == "sources":
        gh = st["gh"]
        gh.run()
        s = gh.mk_psources_maps()
        ps = _view(gh.device_ps_maps()[0], (gh.n_nu, gh.npix), gh.precision == crime_amd.FP64, gh)
        return {"maps": _maps(gh), "sources": ps, "n_sources": s["n_sources"]}
    if kind == "predict":
        return {"cls": st["emu"].predict(st["x"])}
    mlp = st["mlp"]
    mlp.set_params(st["p"])
    loss = mlp.train(st["steps"], st["batch"], 2e-3, 20000, seed=st["seed"] % (1 << 31))
    return {"loss": loss, "params": mlp.params()}


# ---------------------------------------------------------------------------------------------
# the work of a pass: inputs read once, outputs written once, and the arithmetic of the path
# ---------------------------------------------------------------------------------------------
def _mock_work(n, n_side, n_nu, n_sub, fp64):
    e = 8 if fp64 else 4
    n3 = float(n) ** 3
    fft = 2 * 2.5 * n3 * math.log2(n3)              # two real inverse transforms
    cells, samples = 100 * n3, 60 * n3 * n_sub       # lognormal mass and shift; position, redshift, pixel
    return e * n_nu * 12.0 * n_side ** 2, fft + cells + samples


def _sht_flops(n_side, lmax, n_maps):
    nalm = 0.5 * (lmax + 1) * (lmax + 2)
    return n_maps * (4 * nalm * 2 * n_side + 12 * n_side ** 2 * 2.5 * math.log2(4 * n_side))


def work(case):
    kind = case["kind"]
    if kind in ("mock", "training", "power", "sky", "sources"):
        c = dict(dict(n_subcell=0, fp64=False), **_mock_case(case))
        b, f = _mock_work(c["n_grid"], c["n_side"], c["n_nu"], c["n_subcell"] ** 3 or 10, c["fp64"])
        if kind == "training":
            f += _sht_flops(c["n_side"], 3 * c["n_side"] - 1, 16)   # the maps that the pairs name
        if kind == "power":
            n3 = float(c["n_grid"]) ** 3
            b, f = n3 * (16 if c["fp64"] else 8), 7.5 * n3 * math.log2(n3)
        if kind == "sky":
            f += 2 * _sht_flops(c["n_side"], 3 * c["n_side"] - 1, c["n_nu"])
        if kind == "sources":
            b *= 2
        return {"bytes": b, "flops": f}
    if kind == "ensemble":
        got = [0.0, 0.0]
        for k in case["members"]:
            n, s = {"a": (128, 128), "b": (192, 256), "c": (256, 256)}[k]
            b, f = _mock_work(n, s, 64, 10, False)
            got = [got[0] + b, got[1] + f]
        return {"bytes": got[0], "flops": got[1]}
    if kind == "spectra":
        m, lmax, n_side = case["n_maps"], case["lmax"], case["n_side"]
        nalm = 0.5 * (lmax + 1) * (lmax + 2)
        return {"bytes": m * 48.0 * n_side ** 2 + 8.0 * m * m * (lmax + 1),
                "flops": _sht_flops(n_side, lmax, m) + 2.0 * m * (m + 1) * nalm}
    per_row = 2.0 * (8 * 256 + 4 * 256 * 256 + 256)
    if kind == "predict":
        rows = case["cosmologies"] * 2 * case["channels"] * 16
        return {"bytes": 36.0 * rows, "flops": rows * per_row}
    return {"bytes": 4.0 * 2 * 267521 + 40.0 * case["steps"] * case["batch"],
            "flops": 3.0 * case["steps"] * case["batch"] * per_row}


# ---------------------------------------------------------------------------------------------
# the same values in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------
M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox-4x32-10 on int64 tensors that hold 32-bit words."""
    c = [torch.as_tensor(v, dtype=torch.int64, device=DEV) for v in (c0, c1, c2, c3)]
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]     # wraps modulo 2^64; the bits are the product's
        c = [((p1 >> 32) & M32) ^ c[1] ^ k0, p1 & M32, ((p0 >> 32) & M32) ^ c[3] ^ k1, p0 & M32]
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c


def _u53(hi, lo):
    return (((hi << 21) ^ (lo >> 11)) & ((1 << 53) - 1)).double() / 9007199254740992.0


def _array(ptr, n):
    return np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double)), (n,)).copy()


class _Tables:
    """The run description that a handle is made of: radial tables, P(k), channels, sample offsets."""

    def __init__(self, params):
        d = params.desc()
        self.d = d
        for k in ("z_z2r", "r_z2r", "z_r2z", "r_r2z", "d_r2z", "v_r2z"):
            setattr(self, k, torch.from_numpy(_array(getattr(d, k), d.nz)).to(DEV))
        self.logk, self.pk = (torch.from_numpy(_array(p, d.numk)).to(DEV) for p in (d.logk, d.pk))
        self.edges = torch.from_numpy(np.append(_array(d.nu0, d.n_nu), _array(d.nuf, d.n_nu)[-1])).to(DEV)
        self.sub = _array(d.sub_off, 3 * d.n_sub).reshape(-1, 3)
        self.obs = list(d.pos_obs)

    def of_r(self, tab, r):
        i = (r * self.d.idr).long().clamp_(0, self.d.nz - 2)
        return tab[i] + (tab[i + 1] - tab[i]) * (r - self.r_r2z[i]) * self.d.idr


def _fields(t):
    """delta and the velocity potential of a run, [z][y][x]."""
    d, n = t.d, t.d.n_grid
    h = n // 2
    dk = 2 * math.pi / d.l_box
    q = torch.arange(n, device=DEV)
    q = torch.where(q <= h, q, n - q)
    kx, ky = torch.arange(h + 1, device=DEV), torch.arange(n, device=DEV)
    dens = torch.empty((n, n, h + 1), dtype=torch.complex128, device=DEV)
    inv_m = torch.empty((n, n, h + 1), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 24) // (n * (h + 1)))
    for z0 in range(0, n, step):
        z = torch.arange(z0, min(n, z0 + step), device=DEV)
        idx = kx[None, None, :] + (h + 1) * (ky[None, :, None] + n * z[:, None, None])
        w = _philox(idx & M32, idx >> 32, torch.zeros_like(idx), torch.zeros_like(idx), d.seed, 0x47484931)
        mod, ph = torch.sqrt(-torch.log1p(-_u53(w[2], w[3]))), 2 * math.pi * _u53(w[0], w[1])
        m2 = (kx[None, None, :] ** 2 + q[None, :, None] ** 2 + q[z][:, None, None] ** 2).double()
        lgk = 0.5 * torch.log10(m2 * dk * dk)
        i = ((lgk - d.logkmin) * d.idlogk).nan_to_num(0, 0, 0).long().clamp_(0, d.numk - 2)
        amp = torch.sqrt((t.pk[i] + (lgk - t.logk[i]) * (t.pk[i + 1] - t.pk[i]) * d.idlogk) / dk ** 3)
        if d.do_smoothing:
            amp = amp * torch.exp(-0.5 * d.r2_smooth * m2 * dk * dk)
        dens[z] = torch.where(m2 > 0, torch.polar(amp.nan_to_num(0) * mod, ph), 0)
        inv_m[z] = torch.where(m2 > 0, 1 / m2, 0)
    for p in (0, h):   # a real transform keeps the Hermitian part of these planes
        x = dens[:, :, p]
        dens[:, :, p] = 0.5 * (x + torch.roll(torch.flip(x, (0, 1)), (1, 1), (0, 1)).conj())
    norm = (math.sqrt(2 * math.pi) / d.l_box) ** 3 * float(n) ** 3
    vpot = torch.fft.irfftn(dens * inv_m, s=(n, n, n)) * (norm * d.f0h0 / (dk * dk))
    del inv_m
    return torch.fft.irfftn(dens, s=(n, n, n)) * norm, vpot


def _ring_pixels(ns, x, y, z, r):
    """HEALPix RING pixel of directions (Gorski et al. 2005).  A sample on a pixel's edge goes by the last bit:
    the operations of the published routine, in its order."""
    cth = z / r
    za = cth.abs()
    ph = torch.atan2(y, x)
    tt = torch.where(ph < 0, ph + 2 * math.pi, ph) * 0.636619772367581343075535053490057
    tt = torch.where(tt >= 4, 0, tt)
    a, b = ns * (0.5 + tt), ns * cth * 0.75
    jp, jm = torch.floor(a - b).long(), torch.floor(a + b).long()
    ir = ns + 1 + jp - jm
    ip = ((jp + jm - ns + 1 - (ir & 1) + 1) // 2) % (4 * ns)
    belt = 2 * ns * (ns - 1) + (ir - 1) * 4 * ns + ip
    tp = tt - torch.floor(tt)
    tmp = torch.where(za > 0.99, ns * (torch.sqrt(x * x + y * y) / r) / torch.sqrt((1 + za) / 3),
                      ns * torch.sqrt(3 * (1 - za)))
    ir = torch.floor(tp * tmp).long() + torch.floor((1 - tp) * tmp).long() + 1
    ip = torch.floor(tt * ir).long() % (4 * ir)
    cap = torch.where(cth > 0, 2 * ir * (ir - 1) + ip, 12 * ns * ns - 2 * ir * (ir + 1) + ip)
    return torch.where(za <= 2 / 3, belt, cap)


def _mock_exact(params):
    t = _Tables(params)
    d, n, ns = t.d, t.d.n_grid, t.d.n_side
    dens, vpot = _fields(t)
    sigma2 = float((dens * dens).mean() - dens.mean() ** 2)
    npix, dx = 12 * ns * ns, d.l_box / n
    dnu = t.edges[1:] - t.edges[:-1]
    zc = NU_21 / (0.5 * (t.edges[1:] + t.edges[:-1])) - 1
    i = (zc / 0.001).long().clamp(0, d.nz - 2)
    rc = t.r_z2r[i] + (t.r_z2r[i + 1] - t.r_z2r[i]) * (zc - t.z_z2r[i]) / 0.001
    prefac = 90.057156 * d.omega_b * d.hhub * npix / (4 * math.pi) / (rc * rc * dnu)
    maps = torch.zeros(d.n_nu * npix, dtype=torch.float64, device=DEV)
    q = torch.arange(n, device=DEV)
    step = max(1, (1 << 24) // (n * n))
    for z0 in range(0, n, step):
        k = torch.arange(z0, min(n, z0 + step), device=DEV)
        shape = (len(k), n, n)
        x = (dx * (q.double() + 0.5) - t.obs[0])[None, None, :].expand(shape).reshape(-1)
        y = (dx * (q.double() + 0.5) - t.obs[1])[None, :, None].expand(shape).reshape(-1)
        z = (dx * (k.double() + 0.5) - t.obs[2])[:, None, None].expand(shape).reshape(-1)
        v = vpot[k]
        r = torch.sqrt(x * x + y * y + z * z)
        vr = (torch.roll(v, -1, 2) - torch.roll(v, 1, 2)).reshape(-1) * x
        vr += (torch.roll(v, -1, 1) - torch.roll(v, 1, 1)).reshape(-1) * y
        vr += (vpot[(k + 1) % n] - vpot[(k - 1) % n]).reshape(-1) * z
        shift = vr * (0.5 / dx) / r * t.of_r(t.v_r2z, r) if d.rsd else torch.zeros_like(r)
        red = t.of_r(t.z_r2z, r)
        bias = (0.904 + 0.135 * (1 + red) ** 1.696 if d.bias_model == 0 else
                d.bias_b0 + (d.bias_b1 * (1 + red) if d.bias_model == 2 else 0 * red))
        g = t.of_r(t.d_r2z, r) * bias
        mass = dx ** 3 * 0.008 * (1 + red) ** 0.6 * torch.exp(g * (dens[k].reshape(-1) - 0.5 * g * sigma2)) / d.n_sub
        for o in t.sub:
            px, py, pz = x + o[0], y + o[1], z + o[2]
            rs = torch.sqrt(px * px + py * py + pz * pz)
            nu = NU_21 / (1 + t.of_r(t.z_r2z, rs) + shift)
            c = torch.searchsorted(t.edges, nu, right=True) - 1
            ok = (c >= 0) & (c < d.n_nu)
            c = c[ok]
            pix = _ring_pixels(ns, px[ok], py[ok], pz[ok], rs[ok])
            maps.index_add_(0, c * npix + pix, mass[ok] * prefac[c])
    return maps.reshape(d.n_nu, npix), sigma2


class _Rings:
    """Ring geometry and Legendre rows of an Nside, for plain sums over rings."""

    def __init__(self, ns, lmax):
        self.ns, self.lmax, self.npix = ns, lmax, 12 * ns * ns
        i = np.arange(1, 4 * ns)
        north = np.minimum(i, 4 * ns - i)
        cap = north < ns
        self.n = np.where(cap, 4 * north, 4 * ns)
        self.shifted = np.where(cap, 1, (i - ns + 1) & 1)
        self.first = np.concatenate([[0], np.cumsum(self.n)[:-1]])
        z = np.where(cap, 1 - north ** 2 / (3.0 * ns * ns), 4 / 3 - 2 * north / (3.0 * ns))
        self.z = torch.from_numpy(np.where(i > 2 * ns, -z, z)).to(DEV)
        st = np.where(cap, north / ns * np.sqrt((2 - north ** 2 / (3.0 * ns * ns)) / 3.0), np.sqrt(1 - z * z))
        self.st = torch.from_numpy(st).to(DEV)

    def legendre(self, m0, m1):
        """lambda_lm(z_r) for m in [m0, m1): [m - m0][l][ring]."""
        m = torch.arange(m0, m1, device=DEV).double()
        k = np.arange(1, m1)
        log_mm = np.concatenate([[0.0], np.cumsum(0.5 * np.log((2 * k + 1.0) / (2 * k)))]) - 0.5 * math.log(4 * math.pi)
        mm = torch.exp(torch.from_numpy(log_mm[m0:m1]).to(DEV)[:, None] + m[:, None] * torch.log(self.st)[None, :])
        mm = torch.where((m % 2 == 1)[:, None], -mm, mm)
        lam = torch.zeros((m1 - m0, self.lmax + 1, len(self.n)), dtype=torch.float64, device=DEV)
        for ell in range(m0, self.lmax + 1):
            a = torch.sqrt((4.0 * ell * ell - 1) / (ell * ell - m * m).clamp(min=1))
            b = torch.sqrt(((ell - 1.0) ** 2 - m * m).clamp(min=0) / max(1.0, 4.0 * (ell - 1) ** 2 - 1))
            up = torch.zeros_like(mm)
            if ell >= 1:
                low = b[:, None] * lam[:, ell - 2] if ell >= 2 else 0
                up = a[:, None] * (self.z[None, :] * lam[:, ell - 1] - low)
            lam[:, ell] = torch.where((m == ell)[:, None], mm, torch.where((m < ell)[:, None], up, 0))
        return lam

    def blocks(self):
        step = max(1, (1 << 30) // ((self.lmax + 1) * len(self.n)))
        return [(m, min(self.lmax + 1, m + step)) for m in range(0, self.lmax + 1, step)]

    def analyse(self, maps):
        """a_lm of maps [map][pixel] with unit ring weights: [m][l][map]."""
        m = torch.arange(self.lmax + 1, device=DEV)
        f = torch.empty((self.lmax + 1, len(self.n), maps.shape[0]), dtype=torch.complex128, device=DEV)
        host = maps.cpu().numpy()
        for r, n in enumerate(self.n):
            n = int(n)
            # numpy's transforms: a GPU library would compile a plan for each of the ring lengths
            s = torch.from_numpy(np.fft.rfft(host[:, self.first[r]: self.first[r] + n].astype(np.float64))).to(DEV)
            k = m % n
            s = torch.where(k <= n // 2, s[:, torch.minimum(k, n - k)], s[:, torch.minimum(k, n - k)].conj())
            ph = torch.polar(torch.ones(self.lmax + 1, dtype=torch.float64, device=DEV),
                             -math.pi * int(self.shifted[r]) * (m % (2 * n)).double() / n)
            f[:, r] = (s * ph).T
        f *= 4 * math.pi / self.npix
        alm = torch.empty((self.lmax + 1, self.lmax + 1, maps.shape[0]), dtype=torch.complex128, device=DEV)
        for a, b in self.blocks():
            lam = self.legendre(a, b)
            for q in range(a, b):
                alm[q] = torch.complex(lam[q - a] @ f[q].real.contiguous(), lam[q - a] @ f[q].imag.contiguous())
        return alm

    def synthesise(self, alm):
        f = torch.empty((self.lmax + 1, len(self.n), alm.shape[2]), dtype=torch.complex128, device=DEV)
        for a, b in self.blocks():
            lam = self.legendre(a, b)
            for q in range(a, b):
                lt = lam[q - a].T.contiguous()
                f[q] = torch.complex(lt @ alm[q].real.contiguous(), lt @ alm[q].imag.contiguous())
        out = torch.empty((alm.shape[2], self.npix), dtype=torch.float64, device=DEV)
        m = torch.arange(self.lmax + 1, device=DEV)
        f[0] = f[0].real.to(torch.complex128)
        for r, n in enumerate(self.n):
            n = int(n)
            ph = torch.polar(torch.ones(self.lmax + 1, dtype=torch.float64, device=DEV),
                             math.pi * int(self.shifted[r]) * (m % (2 * n)).double() / n)
            s = f[:, r] * ph[:, None]
            d = torch.zeros((n, alm.shape[2]), dtype=torch.complex128, device=DEV)
            d.index_add_(0, m % n, s)
            d.index_add_(0, (-m[1:]) % n, s[1:].conj())
            line = np.fft.irfft(d[: n // 2 + 1].cpu().numpy(), n, axis=0) * n
            out[:, self.first[r]: self.first[r] + n] = torch.from_numpy(line.T.copy()).to(DEV)
        return out


def _weights(alm):
    w = torch.full((alm.shape[0], 1, 1), 2.0, dtype=torch.float64, device=DEV)
    w[0] = 1
    return w


def _cross_cls(alm):
    n, nl = alm.shape[2], alm.shape[1]
    w = _weights(alm)
    out = torch.empty((n, n, nl), dtype=torch.float64, device=DEV)
    for ell in range(nl):
        x = alm[: ell + 1, ell]
        re, im, wl = x.real.contiguous(), x.imag.contiguous(), w[: ell + 1, 0]
        out[:, :, ell] = ((wl * re).T.contiguous() @ re + (wl * im).T.contiguous() @ im) / (2 * ell + 1)
    return out


def _net(p, x):
    """The 8 -> 256 x 5 (SiLU) -> 1 network in 64 bits."""
    h = torch.nn.functional.silu(x @ p[:2048].reshape(8, 256) + p[2048:2304])
    o = 2304
    for _ in range(4):
        h = torch.nn.functional.silu(h @ p[o:o + 65536].reshape(256, 256) + p[o + 65536:o + 65792])
        o += 65792
    return h @ p[o:o + 256] + p[o + 256]


def _train_exact(case, seed):
    x, t, w, p = (torch.from_numpy(v).double().to(DEV) for v in _training_set(case, seed))
    p.requires_grad_(True)
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    rows = torch.arange(case["batch"], device=DEV)
    zero = torch.zeros_like(rows)
    key = int(seed) % (1 << 31)
    for s in range(case["steps"]):
        r = _philox(zero + s, rows, zero, zero, key, 0x4D4C5031)
        n = case["rows"]
        i = ((r[0] % n) * ((1 << 32) % n) + r[1] % n) % n
        e = _net(p, x[i]) - t[i]
        loss = (w[i] * e * e).mean()
        g, = torch.autograd.grad(loss, p)
        losses.append(loss.detach())
        with torch.no_grad():
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            lr = 2e-3 * 0.5 * (1 + math.cos(math.pi * s / 20000))
            p -= lr * (m / (1 - 0.9 ** (s + 1))) / (torch.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
    return {"loss": torch.stack(losses), "params": p.detach()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return [_mock_exact(p)[0] for p in _member_params(case, seed)]
    if kind == "spectra":
        return {"cls": _cross_cls(_Rings(case["n_side"], case["lmax"]).analyse(_sky_maps(case, seed)))}
    if kind == "predict":
        spec = _spec(case)
        x, sc = _network(int(seed), spec, case["cosmologies"])
        p = torch.from_numpy(em.init_params(int(seed))).double().to(DEV)
        z = torch.from_numpy((em.encode(x, sc["dnu"]) - sc["x_mean"]) / sc["x_std"]).to(DEV)
        y = torch.cat([_net(p, b) for b in z.split(1 << 18)])
        return {"cls": sc["scale"] * torch.sinh(sc["y_mean"] + sc["y_std"] * y)}
    if kind == "train":
        return _train_exact(case, int(seed))
    params = _params(_mock_case(case), seed)
    if kind == "power":
        t = _Tables(params)
        n, nbins = t.d.n_grid, t.d.n_grid // 2
        dens = _fields(t)[0]
        sigma2 = float((dens * dens).mean() - dens.mean() ** 2)
        f = torch.fft.rfftn(dens)
        q = torch.arange(n, device=DEV)
        q = torch.where(q <= n // 2, q, n - q)
        kx = torch.arange(n // 2 + 1, device=DEV)
        kk = torch.sqrt((kx[None, None, :] ** 2 + q[None, :, None] ** 2 + q[:, None, None] ** 2).double()).reshape(-1)
        twice = torch.full((n // 2 + 1,), 2.0, dtype=torch.float64, device=DEV)
        twice[0] = twice[-1] = 1
        wt = twice.expand(n, n, -1).reshape(-1)
        b = kk.long()
        ok = b < nbins
        sums = [torch.zeros(nbins, dtype=torch.float64, device=DEV).index_add_(0, b[ok], v[ok] * wt[ok])
                for v in (torch.ones_like(kk), kk, f.abs().square().reshape(-1) * (t.d.l_box ** 3 / float(n) ** 6))]
        return {"k": sums[1] / sums[0] * (2 * math.pi / t.d.l_box), "pk": sums[2] / sums[0], "n": None,
                "sigma2": sigma2}
    maps, sigma2 = _mock_exact(params)
    if kind == "mock":
        return {"maps": maps, "sigma2": sigma2}
    if kind == "sources":   # the sources are random draws: their maps have no closed form
        return {"maps": maps, "sources": None, "n_sources": None}
    if kind == "training":
        spec = _spec(case)
        used = sorted({c for p in spec.pairs for c in p})
        alm = _Rings(spec.n_side, spec.lmax).analyse(maps[used])
        w = _weights(alm)[:, :, 0] / (2 * torch.arange(spec.lmax + 1, device=DEV) + 1.0)
        at = {c: i for i, c in enumerate(used)}
        return {"maps": maps, "cls": torch.stack([(w * (alm[:, :, at[a]] * alm[:, :, at[b]].conj()).real).sum(dim=0)
                                                  for a, b in spec.pairs])}
    fwhm, sig2, mask = _sky(case, seed)
    rings = _Rings(case["n_side"], 3 * case["n_side"] - 1)
    ell = torch.arange(rings.lmax + 1, device=DEV).double()
    beam = torch.exp(-0.5 * (ell * (ell + 1))[:, None] * torch.from_numpy((0.00012352884853326381 * fwhm) ** 2).to(DEV))
    maps = rings.synthesise(rings.analyse(maps) * beam[None])
    pix = torch.arange(rings.npix, device=DEV)
    for c in range(case["n_nu"]):
        w = _philox(pix, pix * 0, pix * 0 + c, pix * 0, int(seed) & M32, 0x4A4F4E54)
        maps[c] += torch.sqrt(-sig2[c] * torch.log1p(-_u53(w[2], w[3]))) * torch.cos(2 * math.pi * _u53(w[0], w[1]))
    return {"maps": maps * torch.from_numpy(mask).to(DEV)}
