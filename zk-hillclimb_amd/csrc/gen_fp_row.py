"""Generate fp_row_consts.inc: the per-lane constants of fp_row.hpp (Fp spread over the 16
lanes of a DPP row as 14 limbs of 28 bits, Montgomery radix R' = 2^392).

  P   the limbs of p
  M   (p n0 + 1) / 2^28 with n0 = -p^-1 mod 2^28: adding m M after dropping a low limb m is
      adding m p n0 and shifting (p n0 = -1 mod 2^28), so m needs no product of its own
  KA  24 p, KB 32 p, in limbs raised by 2^31 (2^30) borrowed from the next limb: KA - b and
      KB - b have no negative limb for the operands the formulas subtract
  IN  2^400 mod p: a row product by it takes R = 2^384 residues to R' form (x 2^8)
  OUT 2^384 mod p: and back (x 2^-8)
Usage: python gen_fp_row.py > fp_row_consts.inc
"""
p = 0x1A0111EA397FE69A4B1BA7B6434BACD764774B84F38512BF6730D2A0F6B0F6241EABFFFEB153FFFFB9FEFFFFFFFFAAAB
L, W = 14, 28
MASK = (1 << W) - 1
PINV = pow(p, -1, 1 << W)
N0 = (1 << W) - PINV


def limbs(v):
    return [(v >> (W * i)) & MASK for i in range(L - 1)] + [v >> (W * (L - 1))]


def raised(v, bit):
    out = [x + ((1 << bit) if i < L - 1 else 0) - ((1 << (bit - W)) if i else 0) for i, x in enumerate(limbs(v))]
    assert sum(x << (W * i) for i, x in enumerate(out)) == v and all(0 < x < 1 << 32 for x in out)
    return out


M = (p * N0 + 1) >> W
assert (p * N0 + 1) & MASK == 0 and M < p
KA, KB = raised(24 * p, 31), raised(32 * p, 30)
TOP = p / 2 ** 364
# KA: up to 8 products (each below 2.96 p, limbs below 2^28 + 16); KB: one value below 31 p with
# limbs below 2^28 + 16
assert all(x >= 8 * ((1 << W) + 16) for x in KA[:-1]) and KA[-1] > 8 * 2.96 * TOP
assert all(x >= (1 << W) + 16 for x in KB[:-1]) and KB[-1] > 31 * TOP + 16
print("// generated by gen_fp_row.py: per-lane constants of the row form of Fp (lanes 14, 15 hold zero)")
print("#define FPR_N0 0x%07xu    // -p^-1 mod 2^28" % N0)
print("#define FPR_PINV 0x%07xu  // p^-1 mod 2^28" % PINV)
for name, v in (("P", limbs(p)), ("M", limbs(M)), ("KA", KA), ("KB", KB), ("IN", limbs(pow(2, 400, p))),
                ("OUT", limbs(pow(2, 384, p))), ("ONE", limbs(pow(2, 392, p)))):
    print("#define FPR_%s_LIMBS %s" % (name, ", ".join("0x%08xu" % x for x in v + [0, 0])))
