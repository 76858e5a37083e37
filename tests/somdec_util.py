"""Carbon and nitrogen inventories of a SomDec (ELM-CN cascade) state, for
the conservation checks of the oracle and of the HIP kernels."""
import numpy as np


def carbon_nitrogen(net, arrays, n):
    """C and N (mol per cell) in the SOM and litter pools and in CO2, NH4+,
    NO3- and N2O, for the first n cells of a state laid out as
    workloads.somdec_workload writes it (SOM1-4, Lit1C-3C, Lit1N-3N)"""
    a = arrays
    sd = net.somdec
    psv = a["porosity"][0, :n] * a["saturation"][0, :n] * 1000.0 * a["volume"][0, :n]
    imm = a["immobile"][:, :n] * a["volume"][0, :n]
    tot = a["total"][:, :n] * psv
    nc_som = sd.arrays["upstream_nc"][3:7]     # SOM1-4 fixed N:C (reactions 4-7)
    C = imm[0:4].sum(0) + imm[4:7].sum(0) + tot[0]
    N = (imm[0:4] * nc_som[:, None]).sum(0) + imm[7:10].sum(0) + tot[1] + tot[2] + 2 * tot[3]
    return C, N


# networks that reach the sandbox's options the ELM-CN workload leaves unused
OPTION_CASES = ("inhibition", "pool-monod", "responses", "scalars", "rates", "ammonium-only",
                "smoothing", "no-smoothing", "linear", "no-split", "trackers")


def option_workload(which, ncell, seed=20261210):
    """an ELM-CN cascade (litter with variable C:N, SOM with fixed C:N) with
    one group of sandbox options, over cells drawn as somdec_workload's"""
    from pfchem import somdec as SD
    from pfchem.network import CellState, ReactionNetwork
    from pfchem.workloads import Workload, somdec_options
    rng = np.random.default_rng(seed)
    prim = ["CO2(aq)", "NH4+", "NO3-", "N2O(aq)", "H+"]
    imm = ["SOM1", "SOM2", "SOM3", "Lit1C", "Lit1N", "Lit2C", "Lit2N"]
    kw, opt = {}, somdec_options()
    mon = [SD.Monod("NH4+", 1.0e-6), SD.Monod("NO3-", 1.0e-6)]
    rx = [dict(upstream="Lit1", downstream=[("SOM1", 0.61)], monod=list(mon)),
          dict(upstream="Lit2", downstream=[("SOM2", 0.3), ("Lit1", 0.2)], monod=list(mon)),
          dict(upstream="SOM1", downstream=[("SOM2", 0.72)]),
          dict(upstream="SOM2", downstream=[("SOM3", 0.4)]), dict(upstream="SOM3")]
    rates = 10.0 ** rng.uniform(-7.5, -5.5, len(rx))
    for r, k in zip(rx, rates):
        r["rate_constant"] = k
    scalars = which == "scalars"
    if which == "inhibition":
        rx[0]["inhibition"] = [SD.Inhibition("NO3-", SD.INHIBITION_THRESHOLD, 1.0e-5, 1.0e5),
                               SD.Inhibition("Lit1C", SD.INHIBITION_INVERSE_MONOD, 0.1)]
        rx[1]["inhibition"] = [SD.Inhibition("CO2(aq)", SD.INHIBITION_MONOD, 1.0e-3)]
        rx[2]["inhibition"] = [SD.Inhibition("SOM1", SD.INHIBITION_MONOD, 0.3),
                               SD.Inhibition("NH4+", SD.INHIBITION_THRESHOLD, 1.0e-5, -1.0e5)]
        rx[3]["inhibition"] = [SD.Inhibition("SOM3", SD.INHIBITION_INVERSE_MONOD, 0.05)]
    elif which == "pool-monod":
        rx[0]["monod"] = [SD.Monod("NH4+", 1.0e-3, 1.0e-8, True), SD.Monod("NO3-", 1.0e-3, 0.0, True)]
        rx[1]["monod"] = [SD.Monod("Lit2C", 0.05, 1.0e-3), SD.Monod("NH4+", 1.0e-6, 2.0e-7)]
        rx[2]["monod"] = [SD.Monod("CO2(aq)", 1.0e-2, 1.0e-7, True), SD.Monod("SOM1", 0.1)]
        rx[3]["monod"] = [SD.Monod("SOM1", 0.5, 0.0, True), SD.Monod("NH4+", 1.0e-6)]
    elif which == "responses":
        for r, (t, q, ea) in zip(rx, [(1, 1.5, 0.0), (3, 2.5, 0.0), (4, 1.5, 5.0e4), (2, 2.0, 0.0),
                                      (0, 1.5, 0.0)]):
            r.update(temperature_response_function=t, Q10=q, Ea=ea)
        rx[0]["moisture_response_function"] = SD.MOISTURE_LOGTHETA
        rx[2]["moisture_response_function"] = SD.MOISTURE_LOGTHETA
        rx[1]["Ox_response_function"] = SD.OX_WFPS
        rx[2]["Ox_response_function"] = SD.OX_WFPS
    elif which == "scalars":
        rx[1].update(temperature_response_function=2, Q10=1.7)
        rx[0]["moisture_response_function"] = SD.MOISTURE_LOGTHETA  # f_w is given: not read
        rx[2]["Ox_response_function"] = SD.OX_WFPS
    elif which == "rates":
        for r in rx[1::2]:
            r["rate_decomposition"] = r.pop("rate_constant")
        rx[0]["rate_ad_factor"] = 5.0
    elif which == "trackers":
        imm += ["HRimm", "Nmin", "Nimm", "Nimp", "NGASmin", "Lit1CHR", "SOM1NMIN", "Lit1NIMM",
                "Lit1NIMP"]
    elif which == "ammonium-only":
        prim = ["CO2(aq)", "NH4+"]
        rx[0]["monod"], rx[1]["monod"] = mon[:1], []
    elif which == "smoothing":
        kw["x0eps"] = 1.0e-4
    elif which == "no-smoothing":
        kw["x0eps"] = 0.0
    elif which == "linear":
        opt = somdec_options(use_log_formulation=False)
    elif which == "no-split":
        kw.update(inhibition_nh4_no3=0.0, n2o_frac_mineralization=0.1)
    pools = [SD.Pool("SOM1", 12.0), SD.Pool("SOM2", 15.0), SD.Pool("SOM3", 15.0), SD.Pool("Lit1"),
             SD.Pool("Lit2")]
    sd = SD.build_somdec(pools, [SD.Reaction(**r) for r in rx], prim, imm, **kw)
    net = ReactionNetwork(primary_species_names=prim, primary_spec_Z=np.zeros(len(prim)),
                          primary_spec_a0=np.zeros(len(prim)), immobile_names=imm, somdec=sd)
    n = ncell
    st = CellState(net, n, somdec_scalars=scalars)
    lu = lambda lo, hi: 10.0 ** rng.uniform(np.log10(lo), np.log10(hi), n)
    draw = {"CO2(aq)": lu(1e-6, 1e-3), "NH4+": lu(1e-7, 1e-4), "NO3-": lu(1e-7, 1e-4),
            "N2O(aq)": np.full(n, 1e-20), "H+": np.full(n, 1e-6)}
    st["total"][:, :n] = np.vstack([draw[p] for p in prim])
    st["pri_molal"][:, :n] = st["total"][:, :n]
    st["pri_act_coef"][:, :n] = 1.0
    for i, name in enumerate(imm):
        st["immobile"][i, :n] = lu(1e-3, 1.0) if name.startswith("SOM") else lu(1e-2, 1.0)
        if name in ("Lit1N", "Lit2N"):
            st["immobile"][i, :n] = (st["immobile"][i - 1, :n] / rng.uniform(20.0, 80.0, n) /
                                     SD.CN_RATIO_MASS_TO_MOL)
        elif i >= 7:  # trackers
            st["immobile"][i, :n] = 1.0e-20
    st["porosity"][0, :n] = rng.uniform(0.3, 0.6, n)
    st["saturation"][0, :n] = rng.uniform(0.2, 1.0, n)
    st["den_kg"][0, :n] = 1000.0
    st["volume"][0, :n] = rng.uniform(0.5, 2.0, n)
    st["temperature"][0, :n] = rng.uniform(-10.0, 35.0, n)
    if scalars:
        st["somdec_f_t"][0, :n] = rng.uniform(0.2, 1.0, n)
        st["somdec_f_w"][0, :n] = rng.uniform(0.0, 1.0, n)
    return Workload("somdec_" + which, net, opt, st, 1800.0, seed, "")
