// Host-side model of the LDS accesses of the forward-only kernel (lncc_forward_kernel.h), for every
// tile width it is built for, from the same lane maps, buffer offsets and step counts the kernel uses
// (lncc_geometry.h). It runs the two roles of a workgroup, F (writes x-sums) and Y (reads rows of
// them), step by step through a sequence of marches of 1, 2, 3, 5 and 8 planes, one after another as a
// workgroup takes its pieces, and checks
//   bounds    every access lies inside Xs, and every Y read at an 8-byte aligned offset;
//   barriers  F and Y pass the same number of barriers in every march;
//   races     between two barriers no float is written by two F units (lanes past the last input row
//             repeat it) or both written and read;
//   coverage  what a counted plane's windows read was written for that plane in the step before:
//             the tile's column x in rows seg * SY + i .. + 2h of the input region, by the F lane
//             that owns the column; every column and row of the tile is some Y lane's, once, and
//             every plane of a march is counted once.
//
// Usage: forward_lds_model [plant]: 1 starts Y on the buffer F writes first, 2 leaves the lanes past
// the last input row unclamped, 3 makes a march one step short, 4 reads rows of a Y lane's neighbour
// column, 5 puts Y's rows one float further; each must be reported.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>
#include <vector>

#include "lncc_geometry.h"

namespace {

int g_plant = 0;
long g_fail = 0;

// prints the first mistake of each kind (the message without its numbers)
void fail(const std::string& what) {
    static std::set<std::string> seen;
    std::string kind;
    for (char c : what)
        if (c < '0' || c > '9') kind += c;
    if (seen.insert(kind).second) std::printf("  FAIL %s\n", what.c_str());
    ++g_fail;
}

// what a float of Xs holds: the input plane (counted over all marches), field, column and row
struct Value {
    int plane = -1, q = -1, col = -1, row = -1;
};

template <int H, int NC>
void check() {
    using G = fl::FwdGeo<H, NC>;
    const long before = g_fail;
    const std::string tag = "h=" + std::to_string(H) + " " + std::to_string(G::RW) + " columns";
    constexpr int SIZE = 2 * G::BUF, NY = G::SY + 2 * H, FL = 64 * G::NFW, YL = 64 * G::NYW;
    std::vector<Value> xs(SIZE);
    std::vector<long> wrote(SIZE, -1), read(SIZE, -1);   // the barrier interval of the last access
    std::vector<int> unit(SIZE, -1);                     // and the F unit of the last write
    long interval = 0, plane0 = 0;

    // the tile's outputs: each (column, segment) is one Y lane's
    std::vector<int> owners(G::RW * G::YSEG, 0);
    for (int yl = 0; yl < YL; ++yl) {
        int seg, x;
        fl::fwd_y_lane<G>(yl, seg, x);
        if (seg < 0 || seg >= G::YSEG || x < 0 || x >= G::RW)
            fail(tag + ": Y lane " + std::to_string(yl) + " outside the tile");
        else
            ++owners[seg * G::RW + x];
    }
    for (int o : owners)
        if (o != 1) fail(tag + ": a column's segment has " + std::to_string(o) + " Y lanes");

    for (const int planes : {1, 2, 3, 5, 8, 1}) {
        const int steps = fl::fwd_steps<G>(planes) - (g_plant == 3 ? 1 : 0);
        int fbuf = G::F_BUF0, ybuf = g_plant == 1 ? G::F_BUF0 : G::Y_BUF0, counted = 0;
        for (int s = 0; s < steps; ++s, ++interval) {
            // F: planes s * PPB + e, those of the march
            for (int e = 0; e < G::PPB; ++e) {
                const int z = s * G::PPB + e;
                if (z >= planes) continue;
                for (int tid = 0; tid < FL; ++tid) {
                    int l, iy;
                    int at = fl::fwd_f_lane<G>(tid, l, iy);
                    if (g_plant == 2) at += (tid >> 4) - iy, iy = tid >> 4;
                    for (int q = 0; q < 5; ++q)
                        for (int j = 0; j < NC; ++j) {
                            const int a = fbuf + e * G::PLANE + q * G::XP + j * 16 * G::XS + at;
                            if (a < 0 || a >= SIZE) {
                                fail(tag + ": F writes out of Xs");
                                continue;
                            }
                            const int u = iy * 16 + l;
                            if (wrote[a] == interval && unit[a] != u) fail(tag + ": Xs[" + std::to_string(a) + "] written by two units");
                            if (iy >= G::IY) fail(tag + ": F lane " + std::to_string(tid) + " writes a row past the input region");
                            wrote[a] = interval;
                            unit[a] = u;
                            xs[a] = Value{(int)(plane0 + z), q, NC * l + j, iy};
                        }
                }
            }
            // Y: every plane of the other buffer, of which those of the march count
            if (s > 0)
                for (int e = 0; e < G::PPB; ++e) {
                    const int z = (s - 1) * G::PPB + e;
                    const bool count = z < planes;
                    counted += count;
                    for (int yl = 0; yl < YL; ++yl) {
                        int seg, x;
                        int at = fl::fwd_y_lane<G>(yl, seg, x) + (g_plant == 5 ? 1 : 0);
                        if (g_plant == 4) at += G::XS;
                        for (int q = 0; q < 5; ++q) {
                            const int a = ybuf + e * G::PLANE + q * G::XP + at;
                            if (a % 2 != 0) fail(tag + ": Y reads at an odd float");
                            for (int i = 0; i < NY; ++i) {
                                if (a + i < 0 || a + i >= SIZE) {
                                    fail(tag + ": Y reads out of Xs");
                                    continue;
                                }
                                read[a + i] = interval;
                                const Value& v = xs[a + i];
                                if (count && (wrote[a + i] != interval - 1 || v.plane != plane0 + z || v.q != q || v.col != x || v.row != seg * G::SY + i))
                                    fail(tag + ": Y lane " + std::to_string(yl) + " reads Xs[" + std::to_string(a + i) + "], which is not its window's");
                            }
                        }
                    }
                }
            for (int a = 0; a < SIZE; ++a)
                if (wrote[a] == interval && read[a] == interval) {
                    fail(tag + ": Xs[" + std::to_string(a) + "] written and read between two barriers");
                    break;
                }
            fbuf = fl::fwd_other<G>(fbuf);
            ybuf = fl::fwd_other<G>(ybuf);
        }
        // F's march, unrolled by 2 k planes, has a barrier after the last plane of each step and passes by
        // whole steps past the end; Y has one barrier a step
        constexpr int K = 2 * H + 1;
        int barriers = 0;
        for (int base = 0; base < steps * G::PPB; base += 2 * K)
            for (int u = 0; u < 2 * K; ++u)
                if (base + u - u % G::PPB < steps * G::PPB && u % G::PPB == G::PPB - 1) ++barriers;
        if (barriers != steps) fail(tag + ": F passes " + std::to_string(barriers) + " barriers, Y " + std::to_string(steps));
        if (counted != planes) fail(tag + ": " + std::to_string(counted) + " of " + std::to_string(planes) + " planes counted");
        plane0 += planes;
    }
    std::printf("forward-only kernel %s: %s\n", tag.c_str(), g_fail == before ? "ok" : "FAILED");
}

}  // namespace

int main(int argc, char** argv) {
    g_plant = argc > 1 ? std::atoi(argv[1]) : 0;
    check<1, 3>();
    check<2, 3>();
    check<3, 3>();
    check<4, 3>();
    check<1, 4>();
    check<2, 4>();
    check<3, 4>();
    std::printf("%s\n", g_fail ? "FAILED" : "all ok");
    return g_fail ? 1 : 0;
}
