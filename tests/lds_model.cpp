// Host-side model of the LDS accesses of the fused LNCC kernel (lncc_fused_kernel.h): for every
// halo h = 1..4 (tile 32 x 32, and 32 x 24 at h = 4), with three adjoint fields (pred gradient)
// and with five (both gradients), it enumerates the LDS reads and writes of every lane in every
// stage from the same role waves, repeated lanes and lane maps the kernel uses (lncc_geometry.h) and
// checks
//   roles     every lane of a role's waves has a unit, and no wave two kinds of unit in one phase
//             (with five adjoint fields AYs units may run on Y waves);
//   bounds    every access lies inside its __shared__ array (spare floats included);
//   races     within a phase no address is written by two units (lanes past a role's last unit
//             repeat that unit, the same values to the same addresses), and no array written in a
//             phase is read in it (the two phases are separated by the workgroup barriers);
//   coverage  every read that feeds a used output (one inside the adjoint region or the output
//             tile) reads an address the producing stage writes, and each used output's window is
//             inside what its lane reads.
// ROCm has no LDS race checker and GPU address sanitizers do not cover LDS, so this stands in
// for the compute-sanitizer workloads of the reference (tests/_sanitize*.py).
//
// Usage: lds_model [plant]. plant = 0 checks the kernel's maps; 1..7 plant one mistake in the
// model's view of them (F writes one column too far, Y rows one float short, AYs stores with a
// row stride one too small, X rows read past their buffer, lanes past the last X unit not sent to
// it, lanes sent to the last Y item but one, an X wave too many), which must be reported. Prints
// one line per configuration and exits 0 when every check passes.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>
#include <vector>

#include "lncc_geometry.h"

namespace {

enum Arr { ZS, XS, GS, GXS, GY, NARR };
const char* kName[NARR] = {"Zs", "Xs", "Gs", "GXs", "GY"};

struct Model {
    int plant = 0;
    long failures = 0;
    std::string cfg;
    std::vector<long> size;
    // per phase: the unit that wrote each address of each array (0 = none), arrays read
    std::vector<std::vector<int>> writes[2];
    std::set<int> read_arrays[2];
    std::set<int> written_arrays[2];

    void fail(const std::string& what) {
        if (failures < 8) std::printf("  FAIL %s: %s\n", cfg.c_str(), what.c_str());
        ++failures;
    }
    void write(int phase, int arr, long addr, int unit) {
        if (addr < 0 || addr >= size[arr]) {
            fail(std::string("write out of ") + kName[arr] + " at " + std::to_string(addr));
            return;
        }
        int& by = writes[phase][arr][addr];
        if (by != 0 && by != unit + 1)
            fail(std::string("address written twice in one phase: ") + kName[arr] + "[" + std::to_string(addr) + "]");
        by = unit + 1;
        written_arrays[phase].insert(arr);
    }
    void read(int phase, int arr, long addr, int len) {
        if (addr < 0 || addr + len > size[arr])
            fail(std::string("read out of ") + kName[arr] + " at [" + std::to_string(addr) + ", " +
                 std::to_string(addr + len) + ")");
        read_arrays[phase].insert(arr);
    }
    // a used read: the addresses [addr, addr+len) must all have been written by the producer
    // (which runs in the other phase)
    void used(int phase, int arr, long addr, int len) {
        for (long a = addr; a < addr + len; ++a)
            if (a < 0 || a >= size[arr] || writes[1 - phase][arr][a] == 0) {
                fail(std::string("used read of unwritten ") + kName[arr] + "[" + std::to_string(a) + "]");
                return;
            }
    }
};

template <int H, int NADJ = 3>
long check(int plant) {
    using G = fl::Geo<H, NADJ>;
    constexpr int NA = G::NADJ;
    Model m;
    m.plant = plant;
    m.cfg = "h=" + std::to_string(H) + " tile 32x" + std::to_string(G::TY) + " " + std::to_string(NA) + " adjoint fields";
    m.size = {5L * G::ZP + G::PAD, 5L * G::XP + G::PAD, (long)NA * G::GP + G::PAD,
              (long)NA * G::GXP + G::PAD, (long)NA * G::GYP};
    for (int p = 0; p < 2; ++p) {
        m.writes[p].resize(NARR);
        for (int a = 0; a < NARR; ++a) m.writes[p][a].assign(m.size[a], 0);
    }
    const int rows_x = fl::row_read(G::SX + 2 * H);                       // X row read (floats)
    const int rows_a = fl::row_read(G::SA + 2 * H);                       // AX row read
    const int rows_y = fl::row_read(G::SY + 2 * H) - (plant == 2 ? 1 : 0);
    const int rows_b = fl::row_read(G::SB + 2 * H);

    // ---- the roles of a lane, and the lane whose unit it takes
    struct Lane {
        bool y, x, b, a, f1;
        int y_lane, x_lane, b_lane, a_lane;
    };
    auto lane_of = [&](int tid) {
        const int wave = tid >> 6;
        Lane l;
        l.y = wave < G::NYW;
        l.x = !l.y && wave < G::NYW + G::NXW + (plant == 7 ? 1 : 0);
        l.b = wave >= G::BL0 / 64 ? wave < G::BL0 / 64 + G::NBW : wave < G::NBYW;
        l.a = false;
        for (int s = 0; s < G::NAW; ++s) l.a = l.a || wave == fl::ax_wave<G>(s);
        l.f1 = G::F_ALL || wave * 64 + fl::NT < G::NIN;
        l.y_lane = std::min(tid, G::Y_LAST - (plant == 6 ? 1 : 0));
        l.x_lane = plant == 5 ? tid : std::min(tid, G::X_LAST);
        l.b_lane = tid >= G::BL0 ? std::min(tid, G::B_LAST) : std::min(tid, G::BY_LAST);
        l.a_lane = wave == fl::ax_wave<G>(G::NAW - 1) ? std::min(tid, fl::ax_last<G>()) : tid;
        return l;
    };
    // ---- writes of both phases first (each phase's reads use the other phase's writes)
    for (int tid = 0; tid < fl::NT; ++tid) {
        const Lane l = lane_of(tid);
        const std::string who = "lane " + std::to_string(tid);
        // P0 / F: the five z-sums of each input column
        for (int j = 0; j < G::J; ++j) {
            if (j > 0 && !l.f1) {
                if (tid + j * fl::NT < G::NIN) m.fail(who + " skips an input column");
                continue;
            }
            const int c = fl::f_lane<G>(tid + j * fl::NT);
            int ix, iy, zaddr;
            if (!fl::f_column<G>(c, ix, iy, zaddr)) {
                if (!G::FPAIR) {
                    m.fail(who + " has no input column");
                    continue;
                }
                // paired stores: a lane without this column writes zeros into the plane padding
                fl::f_column<G>(tid, ix, iy, zaddr);
                zaddr += j * fl::NT;
                if (zaddr < G::IY * G::ZS) m.fail("F padding write inside the plane");
            }
            if (plant == 1) zaddr += 1;
            for (int q = 0; q < 5; ++q) m.write(0, ZS, (long)q * G::ZP + zaddr, c);
        }
        // P1 / Y: the NA adjoint fields of SY outputs of column ax
        if (l.y) {
            int seg, ax, xs, gs;
            if (l.y_lane >= G::YITEMS) m.fail(who + " has no Y item");
            fl::y_item<G>(l.y_lane, seg, ax);
            fl::y_offsets<G>(l.y_lane, xs, gs);  // the kernel's per-lane form of the same addresses
            for (int c = 0; c < NA; ++c)
                for (int i = 0; i < G::SY; ++i) {
                    const int a = gs + c * G::GP + i * G::GST;
                    if (a != fl::y_gs<G>(c, ax, seg * G::SY + i)) m.fail("Y offsets disagree with y_gs");
                    m.write(1, GS, a, l.y_lane);
                }
        }
        int src, dst;
        // P1 / AYs
        if (l.b) {
            if (fl::ays_unit<G>(l.b_lane, src, dst))
                for (int i = 0; i < G::SB; ++i) m.write(1, GY, dst + (long)i * (G::BW - (plant == 3 ? 1 : 0)), l.b_lane);
            else
                m.fail(who + " has no AYs unit");
        }
        // P1 / X, P0 / AX
        if (l.x) {
            if (fl::x_unit<G>(l.x_lane, src, dst))
                for (int i = 0; i < G::SX; ++i) m.write(1, XS, dst + (long)i * G::XS, l.x_lane);
            else
                m.fail(who + " has no X unit");
        }
        if (l.a) {
            if (fl::ax_unit<G>(l.a_lane, src, dst))
                for (int i = 0; i < G::SA; ++i) m.write(0, GXS, dst + (long)i * G::GXS, l.a_lane);
            else
                m.fail(who + " has no AX unit");
        }
        // kinds: a lane has at most one of Y, X, AYs (P1; with five adjoint fields the AYs units run
        // on Y lanes after Y's arithmetic, which reads no LDS row) and at most one of Y, AX (P0)
        if ((l.x && (l.y || l.b)) || (l.y && l.b && !G::B_ON_Y) || (l.y && l.a))
            m.fail(who + " has two units in one phase");
    }

    // ---- reads, and the reads that feed used outputs
    long used_outputs = 0;
    for (int tid = 0; tid < fl::NT; ++tid) {
        const Lane l = lane_of(tid);
        // P0 / Y reads rows of Xs; outputs ay < AY are used, each reading its 2h+1 window
        if (l.y) {
            int seg, ax, xs, gs;
            fl::y_item<G>(l.y_lane, seg, ax);
            fl::y_offsets<G>(l.y_lane, xs, gs);
            const int y0 = seg * G::SY;
            if (xs != ax * G::XS + y0) m.fail("Y row offset disagrees with the item");
            for (int q = 0; q < 5; ++q) {
                const long row = (long)q * G::XP + xs;
                m.read(0, XS, row, rows_y);
                for (int i = 0; i < G::SY; ++i) {
                    if (y0 + i >= G::AY || ax >= G::AX) continue;
                    if (i + 2 * H + 1 > rows_y) m.fail("Y window past the row read");
                    m.used(0, XS, row + i, 2 * H + 1);
                    ++used_outputs;
                }
            }
        }
        // P1 / AYs reads rows of GXs; every output oy < TY is used
        int src, dst;
        if (l.b && fl::ays_unit<G>(l.b_lane, src, dst)) {
            m.read(1, GXS, src, rows_b);
            for (int i = 0; i < G::SB; ++i) {
                m.used(1, GXS, src + i, 2 * H + 1);
                ++used_outputs;
            }
        }
        // P1 / X reads rows of Zs (outputs ax < AX used), P0 / AX reads rows of Gs (all used)
        if (l.x && fl::x_unit<G>(l.x_lane, src, dst)) {
            const long s = src + (plant == 4 ? 5L * G::ZP : 0);
            m.read(1, ZS, s, rows_x);
            const int start = (dst % G::XP) / G::XS;  // first output position of the segment
            for (int i = 0; i < G::SX; ++i) {
                if (start + i >= G::AX) continue;
                m.used(1, ZS, s + i, 2 * H + 1);
                ++used_outputs;
            }
        }
        if (l.a && fl::ax_unit<G>(l.a_lane, src, dst)) {
            m.read(0, GS, src, rows_a);
            for (int i = 0; i < G::SA; ++i) {
                if (i + 2 * H + 1 > rows_a) m.fail("AX window past the row read");
                m.used(0, GS, src + i, 2 * H + 1);
                ++used_outputs;
            }
        }
        // P0 / AZ reads one xy-sum per field of its output column
        if (tid < G::NOUT) {
            int ox, oy;
            fl::az_lane<G>(tid, ox, oy);
            for (int c = 0; c < NA; ++c) {
                const long a = (long)c * G::GYP + oy * G::GYS + ox;
                m.read(0, GY, a, 1);
                m.used(0, GY, a, 1);
                ++used_outputs;
            }
        }
    }
    // ---- phase separation: nothing read in a phase is written in it
    for (int p = 0; p < 2; ++p)
        for (int a : m.read_arrays[p])
            if (m.written_arrays[p].count(a)) m.fail(std::string(kName[a]) + " read and written in one phase");
    std::printf("%s: %ld used outputs checked, %s\n", m.cfg.c_str(), used_outputs,
                m.failures ? "FAILED" : "ok");
    return m.failures;
}

}  // namespace

int main(int argc, char** argv) {
    const int plant = argc > 1 ? std::atoi(argv[1]) : 0;
    long f = 0;
    f += check<1>(plant);
    f += check<2>(plant);
    f += check<3>(plant);
    f += check<4>(plant);
    f += check<1, 5>(plant);
    f += check<2, 5>(plant);
    f += check<3, 5>(plant);
    f += check<4, 5>(plant);
    std::printf("%s\n", f ? "FAILED" : "all ok");
    return f ? 1 : 0;
}
