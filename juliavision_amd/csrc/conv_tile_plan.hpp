// What the one-launch convolution (conv_tile.hip) decides before it launches -- rectangle, chunk, workgroup shape -- and the rule
// its weight loads follow.  Plain C++: a host program checks every load of every choice against the tensor's bounds.
#pragma once
#include <algorithm>
#include <stdint.h>
#include "extents.hpp"

struct ConvShape {
    int Wi, Hi, Cin, N, KW, KH, Cout, OW, OH;
    int sx, sy, px, py, dx, dy, groups, relu;
};

namespace conv_tile {

// Choices are kept by every extent they were made for, each whole: packed two to a word, strides and kernels beyond 65 535 answered
// for one another, and a plan of another stride sends the kernel past its patch.
constexpr int ConvShape::*KEY[] = {&ConvShape::Wi, &ConvShape::Hi, &ConvShape::Cin, &ConvShape::N, &ConvShape::KW, &ConvShape::KH, &ConvShape::Cout, &ConvShape::OW,
                                   &ConvShape::OH, &ConvShape::sx, &ConvShape::sy, &ConvShape::px, &ConvShape::py, &ConvShape::dx, &ConvShape::dy};
inline bool same_shape(const ConvShape &a, const ConvShape &b) {
    for (auto f : KEY)
        if (a.*f != b.*f) return false;
    return true;
}
inline unsigned shape_hash(const ConvShape &a, int cus) {
    unsigned h = (unsigned)cus;
    for (auto f : KEY) h = h * 0x9E3779B1u + (unsigned)(a.*f);
    return h;
}

struct TilePlan {
    int TH, TW, tiles_x, tiles_y;     // output rectangle, rectangles per image
    int CC, nchunk, kc;               // channels a chunk, chunks, CC KH KW
    int ksteps;                       // 16-deep steps of a full chunk
    int PR, PC8, PCL;                 // patch rows, 16-byte pieces a row, halves a row
    int WLD, wpieces;                 // weight row pitch in LDS (halves), 16-byte pieces a row
    int patch_pieces, weight_pieces;  // per chunk
    int tab_off, patch_off, weight_off, stage_bytes;      // LDS layout in bytes: table, then `nbuf` stages of patch + weights
    int nbuf;
};

// Weights travel in 16-byte pieces, eight halves.  Where a chunk or a row leaves fewer, the load is moved back by the rest: into
// the same row, as long as chunk and row have eight halves at all.
constexpr bool weights_by_element(int kc, int CRS) { return kc < 8 || CRS < 8; }
constexpr int weight_back(int left) { return left < 8 ? 8 - left : 0; }
// Where the weights of the chunk from k0 of a row on end: a single chunk, too, may reach past Cin (29 to 31 channels are staged as 32).
constexpr int weight_end(int kc, int CRS, int k0) { return kc < CRS - k0 ? kc : CRS - k0; }
// All pieces that such an end cuts are cut alike: by so many halves the load of one was moved back.
constexpr int weight_cut(int end) { return weight_back(end % 8 ? end % 8 : 8); }

constexpr int LDS_MAX = 160 * 1024;

// The rectangle of `px` pixels with the fewest tiles, then the smallest patch; widths are powers of two so that a wave's
// pixels are whole row pieces.
inline void choose_rectangle(TilePlan &t, const ConvShape &a, int px) {
    int64_t best = INT64_MAX;
    for (int tw = 4; tw <= px; tw *= 2) {
        const int th = px / tw;
        // how far a tile's first column may lie past a multiple of eight: ox0 sx - px is a fixed residue if tw sx is one
        const int slack = tw * a.sx % 8 == 0 ? (int)(((-a.px) % 8 + 8) % 8) : 7;
        const int64_t tiles = ceil_div(a.OW, tw) * ceil_div(a.OH, th);
        const int64_t rows = (int64_t)(th - 1) * a.sy + (a.KH - 1) * a.dy + 1, cols = (int64_t)(tw - 1) * a.sx + (a.KW - 1) * a.dx + 1 + slack;
        const int64_t cost = tiles * (rows * round_up(cols, 8) + px / 2);
        if (cost < best) { best = cost; t.TW = tw; t.TH = th; t.PR = (int)rows; t.PC8 = (int)ceil_div(cols, 8); }
    }
    t.PCL = t.PC8 * 8;
    t.tiles_x = (int)ceil_div(a.OW, t.TW);
    t.tiles_y = (int)ceil_div(a.OH, t.TH);
}

// Chunk depth and LDS layout for `co` output channels and `nt` threads; false where no chunk fits.
inline bool choose_chunk(TilePlan &t, const ConvShape &a, int co, int nt, int parts_bytes) {
    const int taps = a.KH * a.KW;
    auto fits = [&](int cc, bool single) {
        t.CC = cc; t.kc = cc * taps; t.ksteps = (int)ceil_div(t.kc, 16);
        t.wpieces = t.ksteps * 2;                        // whole steps: zero past kc
        t.WLD = t.ksteps * 16 + 8;                       // 16 bytes off a multiple of 32 bytes: rows start in distinct bank groups
        t.patch_pieces = cc * t.PR * t.PC8; t.weight_pieces = co * t.wpieces;
        t.nchunk = (int)ceil_div(a.Cin, cc); t.nbuf = t.nchunk > 1 ? 2 : 1;
        const int64_t patch = round_up(((size_t)cc * t.PR * t.PCL + 8) * 2, 16), weights = (int64_t)co * t.WLD * 2;
        if ((int64_t)cc * t.PR * t.PCL > 65535 || patch + weights > LDS_MAX) return false;
        t.tab_off = 0; t.patch_off = (int)round_up((size_t)t.ksteps * 32, 16);
        t.weight_off = t.patch_off + (int)patch; t.stage_bytes = (int)(patch + weights);
        if (t.patch_off + (int64_t)t.nbuf * t.stage_bytes > LDS_MAX || parts_bytes > LDS_MAX) return false;
        return single || (t.patch_pieces <= 3 * nt && t.weight_pieces <= (co > 64 ? 6 : 5) * nt);
    };
    if (a.Cin <= 16 && fits(a.Cin, true)) return true;
    for (int cc : {64, 32, 16, 8, 4, 2, 1})
        if (cc <= (int)round_up((size_t)a.Cin, 4) && fits(cc, false)) return true;
    return false;
}

struct Shape { int pw, kg, tco; };
constexpr Shape SHAPES[] = {{8, 1, 1}, {8, 1, 2}, {8, 1, 3}, {8, 1, 4}, {8, 1, 5}, {4, 1, 1}, {4, 1, 2}, {4, 1, 3}, {4, 1, 5}, {4, 2, 1}, {4, 2, 2}, {4, 2, 3}, {4, 2, 4}, {2, 4, 1}, {2, 4, 2}, {2, 4, 4}, {2, 2, 1}, {2, 2, 2}};

// Patches that do not overlap: a patch embedding, a strided 1 x 1.
inline bool patches_apart(const ConvShape &a) { return (a.KH - 1) * a.dy < a.sy && (a.KW - 1) * a.dx < a.sx; }
// A patch embedding of channels off sixteen, no deeper than MI_LNA_KMAX: its image (mi_conv2d_f16) and its tokens (mi_conv2d_tokens_f16) have the
// same bits there, those of one chain of sums in the order (ci, kh, kw), which the GEMM over the im2col matrix, unsplit, has either way.
inline bool keeps_one_chain(const ConvShape &a) {
    return a.KW == a.sx && a.KH == a.sy && a.px == 0 && a.py == 0 && a.dx == 1 && a.dy == 1 && a.Cin % 16 && (int64_t)a.Cin * a.KH * a.KW <= MI_LNA_KMAX;
}

// The workgroup shape with the lowest estimate (us), or false where no chunk fits.  Fitted to 130 convolutions in all 18 shapes
// (2 x 2 to 7 x 7, strides 1, 2 and 4, 3 to 384 channels, 16 to 200 000 pixels): the choice is 3 % above the best shape on average.
// A chunk costs its trip to memory and its pieces, a step of a wave its eight gathers and its weight fragments; large outputs 0.1 us a megabyte.
// Too few steps to split (fewer than two a group) go unsplit: 69 such maps take 0.987 of the time of the shape that is estimated lower.
// A margin of 3 % goes to the staged routes (route_of; 1.00 to 1.06 choose alike): on 585 overlapping maps the choice between one launch and
// staging is 1.3 % above the faster, 38 % at worst.
// Patches apart leave little beside the image and the output, which narrow rectangles read and write a sliver of a line at a time, and share
// lines across the dies: 4 / TW us a megabyte of output, all of it 1.1 times; past two workgroups a CU, or deeper than MI_LNA_KMAX in channels the
// patch form takes, twice (2 x 2 over 256 x 256 x 256 -> 64: 45 us, staged 22.6).  844 of them,
// 1 x 1 to 16 x 16: 1.3 % above the faster, 56 % at worst (1 x 768 x 467 x 73 -> 96, 1 x 1 stride 2: 25.4 us in one launch, 39.4 staged).
inline bool choose(const ConvShape &a, int cus, TilePlan &t, Shape &best, double &best_us) {
    if ((int64_t)a.Cout * a.Cin * a.KH * a.KW > INT32_MAX / 2) return false;      // 32-bit offsets
    const bool apart = patches_apart(a), one_chain = keeps_one_chain(a), deep = a.Cin % 16 == 0 && (int64_t)a.Cin * a.KH * a.KW > MI_LNA_KMAX;
    best_us = 1e30;
    TilePlan pick = {};
    for (const Shape &s : SHAPES) {
        TilePlan c = {};
        choose_rectangle(c, a, 32 * s.pw);
        if (!choose_chunk(c, a, 32 * s.tco, s.pw * s.kg * 64, (s.kg - 1) * s.tco * 16 * s.pw * 64 * 4)) continue;
        if (s.kg > 1 && c.nchunk * c.ksteps < 2 * s.kg) continue;
        const int64_t wgs = (int64_t)c.tiles_x * c.tiles_y * ceil_div(a.Cout, 32 * s.tco) * a.N;
        const double rounds = (double)ceil_div(wgs, cus), steps = (double)c.nchunk * c.ksteps * s.pw / 4.0;
        double us = 4.9 + (apart ? 4.0 / c.TW : 0.1) * 2e-6 * (double)a.N * a.Cout * a.OH * a.OW + rounds * (0.3 + 0.147 * s.tco * s.pw + c.nchunk * (0.836 + 0.417e-3 * (c.patch_pieces + c.weight_pieces)) +
                                    steps * (0.027 + 0.0096 * s.tco));
        us *= !apart ? 1.03 : wgs > 2 * cus || deep ? 2.0 : 1.1;
        if (one_chain && (s.kg > 1 || (c.nchunk > 1 && c.kc % 16))) us += 1e6;
        if (us < best_us) { best_us = us; best = s; pick = c; }
    }
    if (best_us >= 1e30) return false;
    t = pick;
    return true;
}

}  // namespace conv_tile
