"""Products around the rule for wrapped transforms (cantor.hpp, wrap_for): the
CPU tests check on which side of it each shape lies, the GPU tests run them."""

# (mp, e, ca, wrapped): a product of 2^mp + e chunk coefficients, ca of one
# operand: one coefficient over, the most that the rule takes and one past it
# (at 2^20 and 2^21 points what the top product costs, at 2^22 a quarter),
# balanced and very unequal operands
PRODUCTS = [(20, 1, 524289, True), (20, 32768, 540673, True), (20, 32769, 540673, False),
            (20, 5, 1000000, True), (21, 3, 2097152, True), (21, 262144, 1300000, True),
            (21, 262145, 1179649, False), (22, 1048576, 2621441, True), (22, 1048577, 2621441, False)]
# (r, residues, wrapped)
SLABS = [(524320, 28, True), (530017, 29, True), (530017, 28, False), (655360, 74, True), (655360, 73, False)]


def chunks(bits):
    return (bits + 31) // 32


def other(mp, e, ca):
    """chunks of the other operand"""
    return (1 << mp) + e + 1 - ca
