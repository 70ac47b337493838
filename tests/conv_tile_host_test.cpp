// The one-launch convolution's choices, made on the CPU by the header its launch code uses (built and run by
// tests/test_conv_tile_plan.py): every 16-byte weight load of every choice lies inside the weight tensor, and what a single chunk's turn into
// is the weight row, zeros behind it.
#include <cstdio>
#include <random>

#include "../juliavision_amd/csrc/conv_tile_plan.hpp"

using namespace conv_tile;

static ConvShape shape(int Wi, int Hi, int Cin, int KW, int KH, int Cout, int sx, int sy, int px, int py, int dx, int dy) {
    ConvShape a = {};
    a.Wi = Wi; a.Hi = Hi; a.Cin = Cin; a.N = 1; a.KW = KW; a.KH = KH; a.Cout = Cout;
    a.sx = sx; a.sy = sy; a.px = px; a.py = py; a.dx = dx; a.dy = dy; a.groups = 1;
    a.OW = (Wi + 2 * px - dx * (KW - 1) - 1) / sx + 1;
    a.OH = (Hi + 2 * py - dy * (KH - 1) - 1) / sy + 1;
    return a;
}

// Halves of the tensor that the load of piece j of a chunk from channel c0 on covers, for output channel co (conv_tile_kernel, weight_load).
static bool inside(const ConvShape &a, const TilePlan &t, int co, int c0, int j) {
    const long taps = a.KH * a.KW, CRS = a.Cin * taps, total = a.Cout * CRS;
    const int left = (int)std::min<long>(t.kc, CRS - c0 * taps) - 8 * j;
    if (left <= 0) return true;
    const long s = co * CRS + c0 * taps + 8 * j;
    if (weights_by_element(t.kc, (int)CRS)) return s >= 0 && s + std::min(left, 8) <= total;
    return s - weight_back(left) >= 0 && s - weight_back(left) + 8 <= total;
}

// Half e of piece j of a single chunk as it is staged: its place in a row, -1 a zero (conv_tile_kernel: weight_load, then the cut).
static int staged(const ConvShape &a, const TilePlan &t, int j, int e) {
    const int CRS = a.Cin * a.KH * a.KW, lim = 8 * j, left = weight_end(t.kc, CRS, 0) - lim;
    if (lim >= t.kc) return -1;
    const int from = left > 0 ? lim - weight_back(left) : 0, wend = weight_end(t.kc, CRS, 0), wgone = weight_cut(wend);
    if (lim >= wend) return -1;
    if (lim + 8 > wend) e += wgone;
    return e < 8 ? from + e : -1;
}

int main() {
    std::mt19937 rng(1);
    auto in = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    int chosen = 0, small = 0, past = 0, bad = 0;
    auto check = [&](const ConvShape &a) {
        TilePlan t;
        Shape s;
        double us;
        if (a.OW < 1 || a.OH < 1 || !choose(a, 256, t, s, us)) return;
        chosen++;
        small += t.kc < 8 && a.Cin * a.KH * a.KW >= 8;
        const int CRS = a.Cin * a.KH * a.KW;
        if (t.nchunk == 1 && !weights_by_element(t.kc, CRS)) {
            past += t.kc > CRS;
            for (int k = 0; k < t.ksteps * 16; k++)
                if (staged(a, t, k / 8, k % 8) != (k < CRS ? k : -1)) {
                    if (!bad++) std::printf("%d -> %d channels, %d x %d on %d x %d: k %d of kc %d, %d a row, is staged from %d\n", a.Cin, a.Cout, a.KH, a.KW, a.Hi, a.Wi, k,
                                            t.kc, CRS, staged(a, t, k / 8, k % 8));
                }
        }
        for (int co : {0, a.Cout - 1})
            for (int ch = 0; ch < t.nchunk; ch++)
                for (int j = 0; j < t.wpieces; j++)
                    if (!inside(a, t, co, ch * t.CC, j)) {
                        if (!bad++) std::printf("%d -> %d channels, %d x %d on %d x %d, stride %d x %d: chunk %d piece %d of kc %d reads outside\n",
                                                a.Cin, a.Cout, a.KH, a.KW, a.Hi, a.Wi, a.sy, a.sx, ch, j, t.kc);
                    }
    };
    check(shape(1414, 637, 64, 1, 3, 6, 5, 6, 0, 1, 1, 1));
    check(shape(1414, 637, 64, 3, 1, 6, 6, 5, 1, 0, 1, 1));
    check(shape(512, 512, 32, 1, 1, 84, 2, 8, 0, 0, 1, 1));
    check(shape(512, 512, 32, 1, 1, 84, 8, 2, 0, 0, 1, 1));
    for (int Cin : {1, 7, 13, 29, 30, 31, 61, 62, 63})
        for (int k : {1, 2, 3, 5}) check(shape(64, 64, Cin, k, k, 32, 1, 1, k / 2, k / 2, 1, 1));
    for (int i = 0; i < 20000; i++) {
        const int KW = in(1, 7), KH = in(1, 7);
        check(shape(in(1, 700), in(1, 700), in(1, 96), KW, KH, in(1, 200), in(1, 12), in(1, 12), in(0, KW / 2), in(0, KH / 2), in(1, 3), in(1, 3)));
    }
    // one output row and column either way, one choice for each
    const ConvShape a = shape(1, 70000, 8, 1, 1, 8, 1, 65537, 0, 0, 1, 1), b = shape(1, 70000, 8, 1, 1, 8, 2, 1, 0, 0, 1, 1);
    if (same_shape(a, b) || !same_shape(a, a)) { std::printf("strides of other calls answer for these\n"); bad++; }
    std::printf("%d choices, %d with chunks under eight halves, %d with a chunk past its row, %d wrong\n", chosen, small, past, bad);
    return bad || !small || !past;
}
