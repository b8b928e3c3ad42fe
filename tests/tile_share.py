"""The choice of tiles and parts for a product (blok_amd/csrc/kx_tile_share.h), compiled for the host."""
import os
import subprocess
from collections import namedtuple

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
# scratch of the hybrid decoder in 32 bits, of it and of Kimi-K2 in bf16: floats, counters
F32, HYBRID, KIMI = (512 * 64 * 128, 512), (256 * 256 * 256, 512), (256 * 256 * 256, 256)
Choice = namedtuple("Choice", "large whole parts tiles")


def build(folder, name="tile_share"):
    """tests/<name>.cpp for the host"""
    exe = str(folder / name)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(os.path.dirname(HERE), "blok_amd", "csrc"),
                        os.path.join(HERE, name + ".cpp"), "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return exe


def _answers(exe, f32, products, scratch):
    block = 32 if f32 else 64
    text = "".join(f"{int(f32)} {t} {r} {c // block} {scratch[0]} {scratch[1]} {CUS}\n" for t, r, c in products)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=300, check=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def choices(exe, f32, products, scratch):
    """products: (tokens, rows, columns)"""
    return [Choice(*a[:4]) for a in _answers(exe, f32, products, scratch)]


def tiles(exe, products, scratch=(0, 0)):
    """"large", "twin" or "medium" for bf16 products"""
    return ["large" if a[0] else "twin" if a[4] else "medium" for a in _answers(exe, False, products, scratch)]


def experts_large(exe, cases):
    """cases: (tokens, top, experts, width, ff); whether their products take tiles of 256 slots where they are not fewer than 96 to an expert"""
    pad = lambda n, to: (n + to - 1) // to * to
    text = "".join(f"{t * top} {e} {2 * pad(ff, 32)} {pad(w, 64) // 64} {w} {pad(ff, 64) // 64} {CUS}\n" for t, top, e, w, ff in cases)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=300, check=True).stdout
    return [line == "1" for line in out.split()]
