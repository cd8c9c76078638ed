// Fused 3D LNCC kernel for gfx950 (MI355X): the loss and the pred gradient, or both gradients.
//
// One workgroup (1024 lanes) owns a TX x TY tile of output columns of one (D,H,W) volume and
// marches along D over a chunk [z0,z1) of planes. Per input plane zi it runs six stages, lagged
// along D so that every quantity is produced from data already on chip:
//
//   F   (registers) lanes own the input columns of the (TX+4h) x (TY+4h) region and keep the
//       last k planes of p, t in a register ring; the z-sums of p, t, p^2, t^2, p*t over planes
//       [zi-k+1, zi] are formed from the ring (below) and written to LDS.
//   X   x-sums of the five z-sums over the (TX+2h)-wide adjoint range.
//   Y   y-sums -> the five k^3 box-sums on the (TX+2h) x (TY+2h) adjoint region; per voxel
//       squared NCC (clamped to 1), loss partial sums, and the adjoint coefficients alpha, beta,
//       gamma (zero where ncc >= 1 or outside the volume).
//   AX  x-sums of alpha, beta, gamma over the TX output columns.
//   AYs y-sums of the three over the TY output rows.
//   AZ  (registers) one lane per output column: a k-deep ring of the xy-sums -> z-sums
//       box(alpha), box(beta), box(gamma), combined with p,t of the output plane (re-read from
//       the L2 as their last use, non-temporal) into the gradient, the only per-voxel write to HBM.
//
// Every box-sum is a sum of its window's own values (lncc_window.h): in x and y blocks of k
// values give each window as a block suffix plus the next block's prefix; along D the march is
// unrolled by k, the ring slot r of plane zi is its position in its block of k planes, and the
// z-sum at zi is the prefix of the current block (planes of slots 0..r, carried in registers)
// plus the suffix of the previous block still in the ring (slots r+1..k-1). So windows of zeros
// sum to exactly zero and windows of one constant to exactly k^3 c, as the reference's direct
// sums do; running sums (add the entering value, subtract the leaving one) would carry the
// rounding of every earlier plane into them.
//
// Software pipeline: the chain F -> X -> Y -> AX -> AYs -> AZ alternates between two phases per
// plane, so each plane costs two workgroup barriers and every LDS buffer is written in one phase
// and read in the other:
//   P0 = {F(zi), Y(zi-1) y-sums, AX(zi-2), AZ(zi-3)}   P1 = {X(zi), Y(zi-1) ncc, AYs(zi-2)}
// Y is split over the phases: its y-sums (LDS reads of Xs) in P0, its ncc and adjoint arithmetic
// (the largest block of VALU work, registers only) in P1, where it runs while the X and AYs units
// wait for their LDS rows. F and AZ run on every lane; the Y items, the X units, the AX units and
// the AYs units sit on waves chosen per phase so that no lane holds two kinds of row at once.
//
// Reference semantics (fused_lncc/csrc/lncc3d.cu:93-107, baselines/torch_lncc.py:25-32):
//   cross = Spt - Sp St/n ; vp = max(Spp - Sp^2/n, 0) + dr ; vt likewise ; ncc = cross^2/(vp vt);
//   ncc >= 1 -> ncc = 1 and zero adjoints; NaN keeps NaN ncc and zero adjoints;
//   A = dncc/dSp, Bc = dncc/dvp, Cc = dncc/dcross; grad = -(1/M)(box A + 2p box Bc + t box Cc).
// The kernel forms the n-fold quantities X = n Spt - Sp St, VP = max(n Spp - Sp^2, 0) + n dr and
// VT likewise (ncc = X^2/(VP VT)): an integer n times a sum and one fused multiply-add, so a
// window of one constant c gives exactly X = 0 and VP - n dr = 0 whenever n^2 c^2 is a float, as
// the reference's Sp St / n division does (a reciprocal 1/n would leave a residue there that the
// division by dr^2 blows up). With r = 1/(VP VT), c = X r, u = c VT, w = St - Sp u it carries
//   alpha = c w, beta = c u, gamma = c   (A = -2 alpha, Bc = -n beta, Cc = 2 n gamma)
// so that grad = (2n/M) (box(alpha)/n + p box(beta) - t box(gamma)).
// Both gradients (MODE_DUAL): the loss is symmetric in p and t, and with u' = c VP, w' = Sp - St u'
// the target's coefficients are alpha' = c w', beta' = c u' and gamma' = c = gamma, so that
// grad_t = (2n/M) (box(alpha')/n + t box(beta') - p box(gamma)): five adjoint fields through the
// adjoint passes instead of three, each formed by the same operations on the same values as in a
// pred-gradient pass over the swapped inputs, so both gradients equal those of two such passes bit
// for bit.
// Range: VP VT = n^2 vp vt would overflow n^2 times earlier than the reference's vp vt (at a
// local standard deviation ~20x smaller at k = 7). The kernel therefore forms VT s instead of VT,
// with s = 2^-E the power of two just below 1/n^2, so that r and c carry a factor 1/s; ncc is
// formed as (X s) (c/s), and alpha, beta, gamma carry 1/s, which the gradient's final scale (2n/M)
// s takes back. Each is one multiply by a literal per voxel (on gfx9 a select or an fma with a
// non-inline constant would need a vector register, and at k >= 5 the kernels are at the
// register limit). Scaling by a power of two is exact, so every result is bit for bit what the
// unscaled arithmetic gives wherever that does not overflow, and VP VT s overflows only where the
// reference's vp vt does (n^2 s lies in (1/2, 1]).
#pragma once
#include "lncc_common.h"
#include "lncc_launch.h"
#include "lncc_lds.h"
#include "lncc_window.h"

namespace fl {

template <int HH, bool BF16, int MODE>
__global__ __launch_bounds__(NT, WG_PER_CU) void lncc_fused_kernel(FusedArgs a) {
    constexpr bool DUAL = (MODE == MODE_DUAL);
    static_assert(MODE == MODE_GRAD || DUAL, "the loss alone and the maps: lncc_forward_kernel.h");
    constexpr int NADJ = DUAL ? 5 : 3;   // adjoint fields
    using G = Geo<HH, NADJ>;
    constexpr int K = G::K;
    constexpr int ELEM = BF16 ? 2 : 4;
    constexpr int J = G::J;
    constexpr int TY = G::TY;

    // one __shared__ array per buffer, so the compiler knows that the reads of one stage do not
    // alias the writes of another and can overlap them
    __shared__ __align__(16) float Zs[5 * G::ZP + G::PAD];
    __shared__ __align__(16) float Xs[5 * G::XP + G::PAD];
    __shared__ __align__(16) float Gs[NADJ * G::GP + G::PAD];
    __shared__ __align__(16) float GXs[NADJ * G::GXP + G::PAD];
    __shared__ __align__(16) float GY[NADJ * G::GYP];
    __shared__ double red[NT / 64];

    const int tid = threadIdx.x;
    // the wave's index in the workgroup, wave-uniform (a scalar register): at k >= 7 the reduction
    // after the march uses it with the lane index (recomputed there), so that no vector register
    // carries the thread index across the march (at the register limit of those kernels it was
    // spilled to scratch: 6 MB of extra HBM traffic per launch at (2,16,128^3)); at k <= 5, where
    // nothing spills, keeping the thread index measured 1% faster
    const int wave_id = __builtin_amdgcn_readfirstlane(tid) >> 6;
    const int D = a.dimD, Hd = a.dimH, Wd = a.dimW;

    // workgroup -> tile. Workgroups go to the 8 XCDs round-robin (workgroup i on XCD i % 8); XCD j
    // takes the j-th contiguous range of logical tiles (q + (j < r) of them, q = nb / 8, r = nb % 8),
    // so that neighbouring tiles, which share halo columns, share one L2
    const uint32_t nb = gridDim.x, bid = blockIdx.x;
    const uint32_t xcd = bid % 8u, q8 = nb / 8u, r8 = nb % 8u;
    uint32_t L = xcd * q8 + min(xcd, r8) + bid / 8u;
    const int tx = (int)(L % (uint32_t)a.ntx); L /= (uint32_t)a.ntx;
    const int ty = (int)(L % (uint32_t)a.nty); L /= (uint32_t)a.nty;
    const int tz = (int)(L % (uint32_t)a.nzc); L /= (uint32_t)a.nzc;
    const int64_t b = (int64_t)L;
    const int x0 = tx * TX, y0 = ty * TY;
    const int z0 = tz * a.dchunk, z1 = min(z0 + a.dchunk, D);
    const int64_t HW = (int64_t)Hd * Wd;
    const uint32_t plane_bytes = (uint32_t)(HW * ELEM);
    const char* pvol = (const char*)a.pred + b * D * HW * ELEM;
    const char* tvol = (const char*)a.target + b * D * HW * ELEM;
    char* const gvol = (char*)a.grad + b * D * HW * ELEM;
    char* const gtvol = DUAL ? (char*)a.grad_t + b * D * HW * ELEM : nullptr;

    // ---- F: per-lane input columns
    uint32_t voff[J];
    int zaddr[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        int ix, iy;
        voff[j] = kOOB;
        if (f_column<G>(f_lane<G>(tid + j * NT), ix, iy, zaddr[j])) {
            const int gx = x0 - 2 * HH + ix, gy = y0 - 2 * HH + iy;
            if (gx >= 0 && gx < Wd && gy >= 0 && gy < Hd) voff[j] = (uint32_t)((gy * Wd + gx) * ELEM);
        }
    }
    if constexpr (G::FPAIR) zaddr[1] = zaddr[0] + NT;
    const bool f_col1 = G::F_ALL || wave_id * 64 + NT < G::NIN;   // this wave has second columns
    // Y items on lanes [0, YITEMS) (y-sums in P0, ncc arithmetic in P1), X and AYs units in P1,
    // AX units in P0 (lncc_geometry.h); offsets into the source and destination buffers
    // (a lane has at most one unit of X and AYs, so the two share one pair of offsets; with five
    // adjoint fields the AYs units sit on Y lanes)
    // The roles are whole waves, a lane past a role's last unit repeats it (lncc_geometry.h).
    const bool wave_y = wave_id < G::NYW;
    const bool wave_x = !wave_y && wave_id < G::NYW + G::NXW;
    const bool wave_b = wave_id >= G::BL0 / 64 ? wave_id < G::BL0 / 64 + G::NBW : wave_id < G::NBYW;
    bool wave_a = false;
#pragma unroll
    for (int sl = 0; sl < G::NAW; ++sl) wave_a = wave_a || wave_id == ax_wave<G>(sl);
    int u_src = 0, u_dst = 0, a_src, a_dst;
    x_unit<G>(min(tid, G::X_LAST), u_src, u_dst);
    {
        constexpr int LAST = ax_last<G>();
        ax_unit<G>((tid >> 6) == ax_wave<G>(G::NAW - 1) ? min(tid, LAST) : tid, a_src, a_dst);
    }
    if (wave_b) ays_unit<G>(tid >= G::BL0 ? min(tid, G::B_LAST) : min(tid, G::BY_LAST), u_src, u_dst);
    int y_seg = 0, y_ax = 0;  // rows seg of AX positions
    // the Y item's offsets into Xs and Gs. At k = 7 they take the registers of the X / AYs unit
    // offsets (a Y lane has no such unit), which with three of Y's rows in flight across F is
    // what keeps the kernel within 128 registers; at the other k separate registers measured
    // faster (k = 9: 1%). With both gradients the Y lanes carry AYs units, whose offsets those are.
    constexpr bool Y_SHARE = HH == 3 && !DUAL;
    int y_xs = 0, y_gs0 = 0;
    if (wave_y) {
        const int item = min(tid, G::Y_LAST);
        y_item<G>(item, y_seg, y_ax);
        if constexpr (Y_SHARE)
            y_offsets<G>(item, u_src, u_dst);
        else
            y_offsets<G>(item, y_xs, y_gs0);
    }
    const int y_xo = Y_SHARE ? u_src : y_xs, y_go = Y_SHARE ? u_dst : y_gs0;
    const int y_start = y_seg * G::SY;
    // per output of the Y segment: inside the volume (ncc and adjoints live) / counted in the loss
    // (inside the volume and in the output tile); the same on every plane
    bool y_inv[G::SY], y_core[G::SY];
    {
        const int gx = x0 - HH + y_ax;
        const bool inx = gx >= 0 && gx < Wd;
        const bool corex = tid < G::YITEMS && y_ax >= HH && y_ax < HH + TX;   // a repeated item counts once
#pragma unroll
        for (int i = 0; i < G::SY; ++i) {
            const int ay = y_start + i, gy = y0 - HH + ay;
            y_inv[i] = inx && gy >= 0 && gy < Hd;
            y_core[i] = y_inv[i] && corex && ay >= HH && ay < HH + TY;
        }
    }
    const bool has_z = tid < G::NOUT;
    int z_ox, z_oy;
    az_lane<G>(tid, z_ox, z_oy);
    const bool z_in = has_z && x0 + z_ox < Wd && y0 + z_oy < Hd;
    const uint32_t z_voff = z_in ? (uint32_t)(((y0 + z_oy) * Wd + x0 + z_ox) * ELEM) : kOOB;

    const int zhi = z1 + 3 + 2 * HH;
    const int zc_lo = max(z0 - HH, 0);
    const int zc_hi = min(z1 + HH, D);
    const int tb = HH + zc_lo;   // the march's first plane: its z windows are the first that X needs

    // F state: the ring of the last k planes' p,t (slot r = position of the plane in its block of
    // k), the prefix sums of the five fields over the current block, and p,t of the next plane
    // (prefetched one step ahead). The march starts with a block: the k - 1 planes before its first
    // one only enter windows, as the previous block, so they are loaded straight into their ring
    // slots, all at once, and cost one memory latency instead of k - 1 steps of the pipeline (chunks
    // of 4 planes at k = 7 took 19 steps, now 13: 96^3 25.2 -> 20.8 us with the drain steps' F left out).
    // LATE: bfloat16 values prefetched for the next step are widened there, not before the barrier that
    // ends this one, where the conversion waits for loads issued a phase ago. (2,16,128^3): k = 5 347 ->
    // 337 us, both gradients at k = 9 981 -> 964 (160x192x224 127 -> 122); k = 9 within 0.5%. At k = 7,
    // where it leaves the registers fuller, 1% slower, at k = 3 within 0.8% either way: as it was.
    constexpr bool LATE = BF16 && (HH == 2 || HH == 4);
    float pring[J][K], tring[J][K], fpre[J][5], fch[J][5], zsum[J][5];
    elem_raw<LATE> pnext[J], tnext[J];
    elem_raw<LATE> pz = 0, tzz = 0;  // AZ: p,t at this step's output plane (prefetched one step ahead)
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            fpre[j][q] = 0.f;
            fch[j][q] = 0.f;
            zsum[j][q] = 0.f;
        }
        pring[j][0] = 0.f;
        tring[j][0] = 0.f;
    }
    {
        const int64_t at = (int64_t)(tb - K + 1) * HW * ELEM;
        uint64_t pa = (uint64_t)(uintptr_t)pvol + at, ta = (uint64_t)(uintptr_t)tvol + at;
#pragma unroll
        for (int r = 1; r <= K; ++r) {   // plane tb - K + r; r = K: the first plane of the march
            const uint32_t n = (uint32_t)(tb - K + r) < (uint32_t)D ? plane_bytes : 0u;
            const rsrc_words rp = words_at(pa, n), rt = words_at(ta, n);
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if (r < K) {
                    pring[j][r < K ? r : 0] = load_elem<BF16>(rp, voff[j]);
                    tring[j][r < K ? r : 0] = load_elem<BF16>(rt, voff[j]);
                } else {
                    pnext[j] = load_raw<BF16, LATE>(rp, voff[j]);
                    tnext[j] = load_raw<BF16, LATE>(rt, voff[j]);
                }
            }
            pa += (uint64_t)HW * ELEM;
            ta += (uint64_t)HW * ELEM;
        }
    }
    // AZ state: the ring of the last k planes' xy-sums of the adjoint fields and their prefix sums
    // over the current block
    float gring[NADJ][K], gpre[NADJ];
#pragma unroll
    for (int c = 0; c < NADJ; ++c) {
        gpre[c] = 0.f;
#pragma unroll
        for (int r = 0; r < K; ++r) gring[c][r] = 0.f;
    }

    double loss_acc = 0.0;
    const float inv_n = a.inv_n, nf = a.nf, ndr = a.ndr;
    constexpr float VS = range_scale(K);   // the range scale s = 2^-E (header)

    // Plane addresses advance by one plane per step, in place: F's next plane zi+1, and AZ's output
    // plane zo = zi-ZO with the plane after it, whose p,t are prefetched. A plane outside its valid
    // range gets a zero-sized resource (its address is never dereferenced).
    constexpr int ZO = 3 + 2 * HH;
    const uint64_t PB = (uint64_t)HW * ELEM;
    const int64_t fz = (int64_t)(tb + 1) * (int64_t)PB, oz = (int64_t)(tb - ZO) * (int64_t)PB;
    uint64_t fpa = (uint64_t)(uintptr_t)pvol + fz, fta = (uint64_t)(uintptr_t)tvol + fz;
    uint64_t opa = (uint64_t)(uintptr_t)pvol + oz + PB, ota = (uint64_t)(uintptr_t)tvol + oz + PB;
    uint64_t oga = (uint64_t)(uintptr_t)gvol + oz, ogta = (uint64_t)(uintptr_t)gtvol + oz;
    const int zn_hi = min(zhi, D);                 // F: new plane zi+1 valid while zi+1 < zn_hi
    // Stage ranges: X(zi) runs for t = zi - HH - zc_lo in [0, nz), Y one step later, AX and AYs two,
    // AZ's input three: one subtraction and one unsigned compare each, zero planes for a wave
    // without the role.
    const uint32_t nz = (uint32_t)(zc_hi - zc_lo);
    const uint32_t n_x = wave_x ? nz : 0u, n_y = wave_y ? nz : 0u, n_a = wave_a ? nz : 0u, n_b = wave_b ? nz : 0u;
    // z-window chains (zstep5 / zstep1): the previous block's sums over ring slots F_CHAIN..K-1
    // (F) and A_CHAIN..K-1 (AZ) kept as partial sums; 0 = none. F's chain (slots 4..6 at k = 7)
    // saves adds but holds five more registers per column; at k = 7 those registers measured
    // better spent on Y's rows in flight across F (three rows and no chain: 2.7% faster than one
    // row and the chain), and at k = 9 they are not there.
    constexpr int F_CHAIN = 0;
    constexpr int A_CHAIN = HH >= 2 && (HH <= 3 || !BF16) ? HH + 1 : 0;

    // Stage bodies; the march below orders them per phase.
    //
    // Y(zi-1): box sums S (y-sums of the rows of the five x-sums), then ncc and the adjoint
    // coefficients at plane zcY (y_math).
    auto y_math = [&](const float (&S)[5][G::SY], int zcY) __attribute__((always_inline)) {
        const bool count = zcY >= z0 && zcY < z1;
        float lsum = -0.f;  // -0 + x == x for every x, so the first add folds away
        float adj[NADJ][G::SY];  // alpha, beta, gamma (and alpha', beta') of the segment's outputs
#pragma unroll
        for (int i = 0; i < G::SY; ++i) {
            const float Sp = S[0][i], St = S[1][i], Spp = S[2][i], Stt = S[3][i], Spt = S[4][i];
            const float X = fmaf(-Sp, St, nf * Spt);
            // n dr is added after the cancellation: folded into the fma that rounds n Spp, it
            // would break that rounding's ties (frequent when n Spp has few significant bits)
            // always upwards, a bias of ~2e-5 in ncc on offset intensities at k = 3
            const float VP = fmaxf(fmaf(-Sp, Sp, nf * Spp), 0.f) + ndr;
            const float VT = (fmaxf(fmaf(-St, St, nf * Stt), 0.f) + ndr) * VS;   // VT s
            const float rr = __builtin_amdgcn_rcpf(VP * VT);
            const float cr = X * rr;             // c / s
            const float ncc = (X * VS) * cr;     // ncc
            const bool live = y_inv[i] && (ncc < 1.0f);
            const float nccc = (ncc >= 1.0f) ? 1.0f : ncc;
            if (y_core[i]) lsum += nccc;
            // masking cr masks all three coefficients (alpha, beta, gamma are multiples of it)
            const float crm = live ? cr : 0.f;
            const float uu = crm * VT;
            const float w = fmaf(-Sp, uu, St);
            adj[0][i] = crm * w;
            adj[1][i] = crm * uu;
            adj[2][i] = crm;
            if constexpr (DUAL) {
                // the target's: u' = (c/s)(VP s), w' = Sp - St u' (the swapped pass's uu, w)
                const float uu2 = crm * (VP * VS);
                adj[3][i] = crm * fmaf(-St, uu2, Sp);
                adj[4][i] = crm * uu2;
            }
            if constexpr (!G::ASWAP) {
#pragma unroll
                for (int c = 0; c < NADJ; ++c) Gs[y_go + c * G::GP + i * G::GST] = adj[c][i];
            }
        }
        if constexpr (G::ASWAP) {  // Gs rows along y: one float4 per field
            static_assert(G::SY == 4, "float4 rows");
#pragma unroll
            for (int c = 0; c < NADJ; ++c)
                lds_store4(Gs + y_go + c * G::GP, adj[c][0], adj[c][1], adj[c][2], adj[c][3]);
        }
        if (count) loss_acc += (double)lsum;
    };
    // F(zi): z-sums of the input region over planes [zi-k+1, zi] (zstep5: the plane prefetched one
    // step ago joins the block prefix and the ring, the previous block's suffix comes from the
    // ring), then the prefetch of the next plane. Every global access of the loop is issued unconditionally
    // (inactive ones through a zero-sized buffer), so the number of outstanding memory operations
    // is the same on every path and the waits before use stay exact. With STORE the z-sums go to
    // the LDS column by column as they are formed; without, f_store writes them later.
    auto f_cols = [&](auto rc, auto store) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        constexpr bool STORE = decltype(store)::value;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (j > 0 && !f_col1) continue;
            zstep5<K, r, F_CHAIN>(widen(pnext[j]), widen(tnext[j]), fpre[j], pring[j], tring[j], fch[j], zsum[j]);
            if constexpr (STORE) {
#pragma unroll
                for (int q = 0; q < 5; ++q) Zs[q * G::ZP + zaddr[j]] = zsum[j][q];
            }
        }
    };
    auto f_pref = [&](int zi) __attribute__((always_inline)) {
        // prefetch plane zi+1
        const uint32_t nb = zi + 1 < zn_hi ? plane_bytes : 0u;
        const rsrc_words rpn = words_at(fpa, nb), rtn = words_at(fta, nb);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            pnext[j] = load_raw<BF16, LATE>(rpn, voff[j]);
            tnext[j] = load_raw<BF16, LATE>(rtn, voff[j]);
        }
        fpa += PB;
        fta += PB;
    };
    auto f_store = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (j > 0 && !f_col1) continue;
#pragma unroll
            for (int q = 0; q < 5; ++q) Zs[q * G::ZP + zaddr[j]] = zsum[j][q];
        }
    };
    // Stage order inside a phase. Each wave runs its stages in program order, so a stage placed
    // between the issue of another stage's LDS reads and their use hides part of their latency.
    //  * P0: AZ's xy-sums are read first. The Y waves issue the reads of Y_EARLY of their five rows
    //    (with the adjoint five at k = 3, three at k = 5, two at k = 7, none at k = 9: more rows held
    //    across F exceed the 128-register budget of a 1024-lane workgroup) and at k <= 5 the AX waves
    //    those of their row; F runs while they arrive (the wait stands at row_take), then the Y waves
    //    read their other rows and form the five box sums, which stay in registers until P1, and the
    //    AX waves their sums; AZ's z-sums and the gradient come last.
    //  * P1: the Y lanes turn their box sums into ncc and the adjoint coefficients (arithmetic
    //    only, no LDS reads: it keeps the SIMDs busy while the rows of the X and AYs units, on the
    //    other waves, arrive), then the X and AYs units (with both gradients, at k >= 5, also on
    //    the first Y lanes: units that do not fit after the X units, 2-7% faster than all AYs
    //    units on Y lanes).
    //  * Both gradients (five adjoint fields, fourteen more ring registers per lane at k = 7):
    //    fewer early rows, all five at k = 3, two (bf16) or none (fp32) at k = 5, none above, and no
    //    AX row before F. At k = 9 the two 9-plane rings and the five adjoint rings exceed the 128
    //    registers even so: 36 (fp32) or 50 (bf16) spill to scratch, and the launch still runs a quarter
    //    faster than two pred-gradient passes. At k = 7 two or four do.
    // What a step costs: 16 waves, 4 per SIMD, none of VALU issue (~55% of the step), LDS (61% active)
    // or HBM (25%) saturated. A scalar instruction takes an issue cycle of its wave like a vector one,
    // and a step had 77 of them for 149 vector ones: lane masks for roles that are whole waves, and
    // five buffer resources rebuilt from 64-bit addresses. Roles as scalar branches and addresses
    // advanced in place leave about 55; with the row waits moved behind F, (2,16,128^3) went from
    // 0.344 / 0.369 / 0.401 / 0.584 to 0.331 / 0.359 / 0.391 / 0.564 ms at k = 3 / 5 / 7 / 9.
    constexpr int Y_EARLY = DUAL ? (HH <= 1 ? 5 : HH == 2 ? (BF16 ? 2 : 0) : 0)
                                 : HH <= 1 ? 5 : HH == 2 ? 3 : HH == 3 ? 2 : 0;   // Y rows read before F
    constexpr bool F_STORE_AT_ONCE = Y_EARLY < 5;
    // no z-sums for the drain steps, which X does not read (2-5% at k >= 5; at k = 3 1% slower, and both
    // gradients at k = 9, which spill, 8%). What it costs: with the branch around F in the march, taken or
    // not, float32 planes of 256 x 256 at k = 7 are read from HBM 1.6 times instead of 1.05 (AZ's re-read
    // misses the L2): (2,16,256^3) 3.00 -> 3.09 ms, both gradients 3.71 -> 3.79; (1,1,160,192,224) 55.2
    // -> 54.2 us, 96^3 21.4 -> 20.8, bfloat16 faster at every size.
    constexpr bool F_STOP = HH >= 2 && !(DUAL && HH == 4);
    constexpr bool AX_EARLY = HH <= 2 && !DUAL;               // the AX row read before F
    constexpr int NY = G::SY + 2 * HH, NA = G::SA + 2 * HH, NX = G::SX + 2 * HH, NB = G::SB + 2 * HH;
    // P0's early reads (Y's first rows or the AX row) share one register array: the two kinds of
    // lane sit on different waves
    constexpr int YQ = row_quads(NY);
    constexpr int NEQ = cmax(cmax(Y_EARLY * YQ, AX_EARLY ? row_quads(NA) : 0), 1), NEH = cmax(Y_EARLY, 1);

    for (int base = tb; base < zhi; base += K) {
        static_for<0, K>([&](auto rc) __attribute__((always_inline)) {
            const int zi = base + decltype(rc)::value;
            if (zi >= zhi) return;
            const int zcY = zi - 1 - HH;   // the plane Y(zi-1) is centred on (the z-sums of F(z): z-h)
            const uint32_t t = (uint32_t)(zi - tb);
            const bool do_x = t < n_x, do_y = t - 1u < n_y, do_a = t - 2u < n_a, do_b = t - 2u < n_b;
            const bool actA = t - 3u < nz;   // the xy-sums AZ(zi-3) reads

            // ============================ phase P0 ============================
            // AZ(zi-3) reads, Y(zi-1) y-sums, AX(zi-2), F(zi), AZ(zi-3)
            // AZ's xy-sums: read first, except at k = 9, where they would be held across F
            float ys[NADJ];
            auto az_read = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int c = 0; c < NADJ; ++c) {
                    // read whatever actA says (the value is dropped when it is false), so that the
                    // three reads pair up
                    const float gy = GY[c * G::GYP + z_oy * G::GYS + z_ox];
                    ys[c] = actA ? gy : 0.f;
                }
            };
            if constexpr (HH <= 3) az_read();
            lds_f4 eq[NEQ];
            lds_f2 eh[NEH];
            if (do_y) {
#pragma unroll
                for (int q = 0; q < Y_EARLY; ++q) row_load<NY>(Xs + q * G::XP + y_xo, eq + q * YQ, eh[q]);
            } else if (AX_EARLY && do_a) {
                row_load<NA>(Gs + a_src, eq, eh[0]);
            }
            float S[5][G::SY];  // Y's box sums, carried into P1
            if (!F_STOP || t < nz) f_cols(rc, std::integral_constant<bool, F_STORE_AT_ONCE>{});
            f_pref(zi);
            if (do_y) {
                // the early rows (held in eq, eh), the rest read now
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    float v[NY];
                    if (q < Y_EARLY) {
                        row_take<NY>(eq + q * YQ, eh[q < Y_EARLY ? q : 0], v);
                    } else {
                        lds_row(Xs + q * G::XP + y_xo, v);
                    }
                    box_sums<HH, G::SY>(v, S[q]);
                }
            } else if (do_a) {
                // AX(zi-2): x-sums (y-sums with ASWAP) of one of alpha, beta, gamma over one segment
                float v[NA], o[G::SA];
                if constexpr (AX_EARLY) {
                    row_take<NA>(eq, eh[0], v);
                } else {
                    lds_row(Gs + a_src, v);
                }
                box_sums<HH, G::SA>(v, o);
#pragma unroll
                for (int i = 0; i < G::SA; ++i) GXs[a_dst + i * G::GXS] = o[i];
            }
            if constexpr (!F_STORE_AT_ONCE) f_store();
            if constexpr (HH > 3) az_read();
            {
                // AZ(zi-3): z-sums of the xy-sums over the k planes of the output plane zo = the
                // prefix of the current block plus the previous block's suffix (ring and chain)
                // (lanes without an output column run on a clamped one and store out of range,
                // i.e. nothing)
                constexpr int r = decltype(rc)::value;
                float gw[NADJ];
#pragma unroll
                for (int c = 0; c < NADJ; ++c) gw[c] = zstep1<K, r, A_CHAIN>(ys[c], gpre[c], gring[c]);
                const int zo = zi - ZO;
                const float po = widen(pz), to = widen(tzz);
                const float g = a.gscale * fmaf(inv_n, gw[0], fmaf(po, gw[1], -to * gw[2]));   // gscale holds s
                // Non-temporal: the gradient is never read back, and this re-read of p,t is the
                // last use of those lines. With the default policy both would be promoted in the
                // L2 and push out the planes that F loaded and this stage re-reads 2h+3 steps
                // later, so that every input byte would be fetched about twice; marked
                // evict-first, every input byte is fetched from HBM once at (2,16,128^3) (float32
                // planes of 256 x 256: F_STOP above). bf16 gradient rows of a tile are half a
                // 128-byte line (the x-neighbour tile writes the other half): those stores keep the
                // default policy, so that the L2 merges the two halves into one write.
                const uint32_t gb = zo >= z0 ? plane_bytes : 0u;   // zo < z1 up to the march's last step
                store_elem_buf<BF16, BF16 ? 0 : kNT>(words_at(oga, gb), z_voff, g);
                oga += PB;
                if constexpr (DUAL) {
                    const float gt = a.gscale * fmaf(inv_n, gw[3], fmaf(to, gw[4], -po * gw[2]));
                    store_elem_buf<BF16, BF16 ? 0 : kNT>(words_at(ogta, gb), z_voff, gt);
                    ogta += PB;
                }
                // prefetch p,t at the next step's output plane; issued after this step's use, so
                // one register each suffices and no copy has to wait for the load
                const uint32_t ob = (uint32_t)(zo + 1 - z0) < (uint32_t)(z1 - z0) ? plane_bytes : 0u;
                pz = load_raw<BF16, LATE, kNT>(words_at(opa, ob), z_voff);
                tzz = load_raw<BF16, LATE, kNT>(words_at(ota, ob), z_voff);
                opa += PB;
                ota += PB;
            }
            __syncthreads();

            // ============================ phase P1 ============================
            // Y(zi-1) ncc arithmetic, X(zi), AYs(zi-2)
            if (do_y) y_math(S, zcY);
            if (do_x) {
                // X(zi): x-sums of one of the five z-sums over one segment (feeds Y at the next plane)
                float v[NX], o[G::SX];
                lds_row(Zs + u_src, v);
                box_sums<HH, G::SX>(v, o);
#pragma unroll
                for (int i = 0; i < G::SX; ++i) Xs[u_dst + i * G::XS] = o[i];
            } else if (do_b) {
                // AYs(zi-2): y-sums (x-sums with ASWAP) of one of alpha, beta, gamma at plane zcB
                float v[NB], o[G::SB];
                lds_row(GXs + u_src, v);
                box_sums<HH, G::SB>(v, o);
#pragma unroll
                for (int i = 0; i < G::SB; ++i) {
                    if constexpr (G::ASWAP) {  // GY rows along x: float4s
                        if (i % 4 == 0)
                            lds_store4(GY + u_dst + i, o[i], o[i + 1], o[i + 2], o[i + 3]);
                    } else {
                        GY[u_dst + i * G::BW] = o[i];
                    }
                }
            }
            __syncthreads();
        });
    }

    // ---- workgroup partial of the ncc sum: wave64 reduction, then the waves in fixed order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off, 64);
    const int lane = HH >= 3 ? (int)__lane_id() : (tid & 63);
    const int wave = HH >= 3 ? wave_id : (tid >> 6);
    if (lane == 0) red[wave] = loss_acc;
    __syncthreads();
    if (wave == 0 && lane == 0) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) sum += red[w];
        a.partials[bid] = sum;
    }
}

template <int HH>
hipError_t launch_fused(int mode, bool bf16, const FusedArgs& a, uint32_t nblocks, hipStream_t st) {
    const dim3 grid(nblocks), block(NT);
#define FL_LAUNCH(BF, MD) hipLaunchKernelGGL((lncc_fused_kernel<HH, BF, MD>), grid, block, 0, st, a)
    if (mode == MODE_GRAD) {
        if (bf16) FL_LAUNCH(true, MODE_GRAD); else FL_LAUNCH(false, MODE_GRAD);
    } else if (mode == MODE_DUAL) {
        if (bf16) FL_LAUNCH(true, MODE_DUAL); else FL_LAUNCH(false, MODE_DUAL);
    } else {
        return hipErrorInvalidValue;
    }
#undef FL_LAUNCH
    return hipGetLastError();
}

}  // namespace fl
