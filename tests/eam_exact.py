"""The closed forms of the Pd-H potential (potential.cpp:16-205) in 50 digits, with
the constants as the doubles a program reads, and forward derivatives."""
from decimal import Decimal, getcontext

F_PD, F_H, PHI_PD, PHI_PDH, PHI_HH = range(5)  # the r-functions, in the order of a2c_eam_tables
getcontext().prec = 50


def D(x):
    return Decimal(float(x))


class Dual:
    """value and slope in 50 digits"""

    def __init__(self, v, d=Decimal(0)):
        self.v, self.d = (v if isinstance(v, Decimal) else D(v)), d

    def __add__(self, o):
        o = o if isinstance(o, Dual) else Dual(o)
        return Dual(self.v + o.v, self.d + o.d)

    __radd__ = __add__

    def __neg__(self):
        return Dual(-self.v, -self.d)

    def __sub__(self, o):
        return self + (-(o if isinstance(o, Dual) else Dual(o)))

    def __mul__(self, o):
        o = o if isinstance(o, Dual) else Dual(o)
        return Dual(self.v * o.v, self.d * o.v + self.v * o.d)

    __rmul__ = __mul__

    def exp(self):
        e = self.v.exp()
        return Dual(e, e * self.d)

    def log(self):
        return Dual(self.v.ln(), self.d / self.v)

    def sqrt(self):
        s = self.v.sqrt()
        return Dual(s, self.d / (2 * s))


def tail(r, amplitude, decay, start):
    return amplitude * ((r - start) * Dual(D(decay) / D(amplitude))).exp()


def f_pd(r):
    t = r * 0.2
    if t.v * 5 > 5:
        return tail(t * 5.0, 0.001510569378297, -0.077976566126292, 5.0)
    p = t
    for b, c in ((2.7267629107325706, 1.8716766113599643), (2.50290548851635, 1.668549182690922),
                 (2.0924467509943674, 1.3150372774478005), (1.564328475106985, 0.8987511149780485),
                 (1.009780903403673, 0.5124363774128722), (0.5304054524800665, 0.2169886022464641),
                 (0.1356566408715063, 0.035852347523891395)):
        p = p * (t * (t - b) + c)
    return -0.02972698211669922 + t * (0.6676807403564453 + t * (-255.8965835571289 + t * (
        14673.409149169922 + -2.597301181336601e7 * p)))


def phi_pd(r):
    t = r * 0.2
    if t.v * 5 > D(5.05):
        return tail(t * 5.0, -0.016958780164980, 0.089019679316328, 5.05)
    p = -79415.24035137112 * (t - 1.0699996145674568) * (t - 1.06015072612581) * (t - 0.42433991011376526) * (
        t + 0.06169160085238687)
    for b, c in ((2.0586473420376348, 1.0683922574015199), (1.6696359816422877, 0.7337878627470482),
                 (1.1690370066230809, 0.3909805777737639), (0.2635598721249787, 0.033551116514910245)):
        p = p * (t * (t - b) + c)
    return p + 2 * 0.251546 * f_pd(r)


def f_h(r):
    if r.v > D(5.35):
        return tail(r, 0.009986990526578, -0.013075667086408, 5.35)
    return 11.0025 * (-1.30927 * r).exp()


def morse(r, a, d, depth, al, be, r0):
    if r.v > D(5.35):
        return tail(r, a, d, 5.35)
    return depth * (be * (-al * (r - r0)).exp() - al * (-be * (r - r0)).exp())


R_FUNCTIONS = {
    F_PD: f_pd, F_H: f_h, PHI_PD: phi_pd,
    PHI_PDH: lambda r: morse(r, -3.353001113951400e-04, 7.147062196813336e-04, 0.2494540, 4.82613, 2.13158, 1.50964),
    PHI_HH: lambda r: morse(r, -0.003702722457147, 0.005465945471933, 0.0661496, 3.67263, 1.47797, 2.51980)}


def embed_pd(rho):
    r = rho * Dual(1 / Decimal(50))
    p = 295878.9003038662 * (r - 0.20581955357385892) * (r - 0.081228755904399) * r * (r + 0.05298811034615951)
    for b, c in ((2.4242616904962846, 1.4791899886249564), (2.1376274623740064, 1.2169215689822592),
                 (1.6486007989726832, 0.8159825255339774), (1.0749204110338482, 0.42007491336688396),
                 (0.5128056047933808, 0.12468685331167456)):
        p = p * (r * (r - b) + c)
    return p - 50.0 * 0.251546 * r


def embed_h(rho):
    c, d, a, b = D(0.000197047), D(1.18860), D(9.99780), D(60.0155)
    u = rho + 0.0540638
    pd = (u.log() * Dual(d)).exp()
    p = pd * u
    return (p * u * Dual(1 / (2 + d)) - p * Dual((a + b) / (1 + d)) + pd * Dual(a * b / d)) * Dual(-c) + 0.0296604 * rho
