"""Lengths whose factorings hold every radix in every place the mixed-radix kernel is given it."""

LENGTHS = [20, 21, 24, 25, 26, 32, 140, 192, 242, 864, 1715, 2145, 2560, 2925, 3375, 4000, 4374, 5346, 7056]
