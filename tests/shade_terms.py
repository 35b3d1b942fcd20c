"""How far sums of the shading adjoint's terms may lie apart when the same terms are added in another order."""
import numpy as np


def dot(a, b):
    return (a * b).sum(-1)


def unit(a):
    return a / np.linalg.norm(a, axis=-1, keepdims=True)


def order_bounds(model, rec, color, target):
    """Per element of the albedo, roughness and intensity gradients of these records: a bound on the difference of two
    FP32 sums of its terms.  An element of n terms takes at most n - 1 roundings of 2^-24 of the sum of the terms'
    magnitudes on either side; of many terms they fall either way, so 16 sqrt(n) stands in for 2 n where it is less."""
    albedo = model.d_albedo.download().astype(np.float64).reshape(-1, 3)
    rough = model.d_rough.download().astype(np.float64)
    lights = model.d_lpos.download().astype(np.float64).reshape(-1, 3)
    power = model.d_inten.download().astype(np.float64)
    live = rec["tri0"] >= 0
    rec = rec[live]
    g = 2.0 * np.abs(color.astype(np.float64).reshape(-1, 3) - target.astype(np.float64).reshape(-1, 3))[live]
    t0, again = rec["tri0"], rec["tri1"] >= 0
    t1 = np.where(again, rec["tri1"], 0)
    p, n, eye, q, nq = (rec[k].astype(np.float64) for k in ("p", "n", "eye", "q", "nq"))
    a0, r = albedo[t0], rough[t0]
    a1 = np.where(again[:, None], albedo[t1], 0.0)
    direct, slope, second = np.zeros(len(rec)), np.zeros(len(rec)), np.zeros(len(rec))
    inten, inten_n = np.zeros(len(power)), np.zeros(len(power))
    for l, (light, intensity) in enumerate(zip(lights, power)):
        seen_p, seen_q = ((rec["vis"] >> np.uint32(b + l)) & 1 != 0 for b in (0, 16))
        lo, li = unit(eye - p), unit(light - p)
        lh = unit(li + lo)
        c_o, c_i, c_h = (np.maximum(dot(n, v), 0.0) for v in (lo, li, lh))
        f = 0.04 + 0.96 * (1.0 - np.maximum(dot(lh, lo), 0.0)) ** 5
        a2 = r ** 4
        den = c_h ** 2 * (a2 - 1.0) + 1.0
        d = a2 / (np.pi * den ** 2)
        d_d = np.abs(den - 2.0 * a2 * c_h ** 2) / (np.pi * den ** 3) * 4.0 * r ** 3
        k = (r + 1.0) ** 2 / 8.0
        d_i, d_o = c_i * (1.0 - k) + k, c_o * (1.0 - k) + k
        s_i, s_o = c_i / d_i, c_o / d_o
        d_g = (c_i * (1.0 - c_i) / d_i ** 2 * s_o + s_i * c_o * (1.0 - c_o) / d_o ** 2) * (r + 1.0) / 4.0
        scale = np.maximum(1e-5, 4.0 * c_i * c_o)
        A = intensity / dot(light - p, light - p) * c_i
        diffuse, specular = A * (1.0 - f), A * f * d * s_i * s_o / scale
        direct += np.where(seen_p, diffuse, 0.0)
        slope += np.where(seen_p, A * f * (d_d * s_i * s_o + d * d_g) / scale, 0.0)
        b = intensity / np.maximum(dot(light - q, light - q), 1e-30) * np.clip(dot(nq, unit(light - q)), 0.0, 1.0)
        b = np.where(seen_q, b, 0.0)
        second += b
        inten[l] = (np.where(seen_p, dot(g, diffuse[:, None] * a0 + specular[:, None]), 0.0) +
                    dot(g, a0 * a1) * b).sum() / intensity
        inten_n[l] = 2 * (seen_p | seen_q).sum()
    size = np.zeros((len(rough), 3)), np.zeros(len(rough)), inten
    count = np.zeros((len(rough), 3)), np.zeros(len(rough)), inten_n
    np.add.at(size[0], t0, g * (direct[:, None] + a1 * second[:, None]))
    np.add.at(size[0], t1[again], (g * a0 * second[:, None])[again])
    np.add.at(size[1], t0, g.sum(1) * slope)
    np.add.at(count[0], t0, 1.0)
    np.add.at(count[0], t1[again], 1.0)
    np.add.at(count[1], t0, 1.0)
    # 1.01: the magnitudes are those of the exact terms, not of the FP32 ones
    return [(1.01 * np.minimum(2.0 * n, 16.0 * np.sqrt(n)) * 2.0 ** -24 * s).reshape(-1) for s, n in zip(size, count)]
