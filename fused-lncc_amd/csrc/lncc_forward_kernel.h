// Forward-only LNCC kernel for gfx950 (the loss without a gradient, and the per-voxel maps).
//
// Without the adjoint a tile needs a halo of h instead of 2h, and no ring of adjoint sums holds
// registers. One workgroup owns a tile of rows of one volume, marches along D over [z0, z1), and
// splits its waves into two roles that meet in LDS once per plane:
//
//   F  lanes own NC consecutive input columns each, 16 lanes (a DPP row) per input row, 4 rows per
//      wave: the z-sums of p, t, p^2, t^2, pt from a register ring of the last k planes, then the x
//      window sums across the DPP row without LDS: a window is a suffix of the left lane's columns
//      (at k = 9 of the two left lanes'), a part of the own ones and a prefix of the right lane's.
//   Y  lanes own one column and four output rows: the y window sums of the five x-sums -> the box
//      sums, ncc, the loss partial or the maps of four voxels.
//
// F writes one of two LDS buffers while Y reads the other, one barrier for PPB planes.
// The DPP row is the tile's width RW = 16 NC: a row's first and last h columns lack a neighbour, so
// neighbouring tiles overlap by 2h columns; at the volume's edges the missing neighbours are zeros,
// which is what the window wants, and nothing is lost (RW columns hold a volume of W <= RW whole).
//
// Window sums, formula, clamp, NaN policy and range scale are those of lncc_fused_kernel.h: every
// sum is one of its window's own values.
//
// Bound: VALU issue. At k = 7 a plane of a 48 x 32 tile takes 2045 cycles of a CU (counters at
// (2,16,128^3)); its 115 vector instructions a wave fill ~1550 of them per SIMD at their measured issue
// rates (additions and products 2.3 cycles, DPP additions, max, compares and selects 4.2, the reciprocal
// 8), 91% as SQ_ACTIVE_INST_VALU counts them (four cycles each); the LDS is active for 862; HBM fetches
// 1.036 / 1.056 / 1.076 / 1.100 times the input bytes at k = 3 / 5 / 7 / 9. At (2,16,128^3) fp32: 0.219 / 0.242 / 0.281 / 0.452 ms -> 0.150 / 0.164 / 0.179 /
// 0.216 ms at k = 3 / 5 / 7 / 9 against the gradient kernel run without its adjoint, whose x pass
// goes through LDS and whose tile carries the adjoint's halo (3.0 TB/s of 8 B per voxel at k = 7);
// the map of 160x192x224 at k = 9 0.0556 -> 0.0356 ms. F is the longer role and has the lower wave
// indices, which the SIMDs serve first (Y first: 9% slower at k = 7).
#pragma once
#include "lncc_common.h"
#include "lncc_launch.h"
#include "lncc_window.h"
#include "lncc_lds.h"

namespace fl {

// The value of the lane D to the left (D < 0) or right of its DPP row, 0 past the row's ends.
template <int D>
__device__ __forceinline__ float row_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), D < 0 ? 0x110 - D : 0x100 + D, 0xF, 0xF, true));
}
// x window sums of NC columns per lane across a DPP row: out[j] = sum of columns j-h .. j+h of the
// row, zero past its ends. One addition per prefix and suffix, one per neighbour (v_add_f32_dpp).
template <int HH, int NC>
__device__ __forceinline__ void xsum_row(const float (&v)[NC], float (&out)[NC]) {
    static_assert(HH < 2 * NC, "windows reach two lanes each way at most");
    float pre[NC + 1], suf[NC + 1];   // sums of the first / last m columns
    pre[1] = v[0];
    suf[1] = v[NC - 1];
#pragma unroll
    for (int m = 2; m <= NC; ++m) {
        pre[m] = pre[m - 1] + v[m - 1];
        suf[m] = m == NC ? pre[m] : v[NC - m] + suf[m - 1];
    }
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const int left = HH - j, right = j + HH - (NC - 1);   // columns needed left and right of the own ones
        float s = left >= 0 ? pre[right >= 0 ? NC : j + HH + 1] : suf[NC + left];
        if (left > 0) s += row_lane<-1>(suf[left < NC ? left : NC]);
        if (right > 0) s += row_lane<1>(pre[right < NC ? right : NC]);
        if (left > NC) s += row_lane<-2>(suf[left - NC]);
        if (right > NC) s += row_lane<2>(pre[right - NC]);
        out[j] = s;
    }
}

// A row of NV floats (even) at an 8-byte aligned LDS address as 64-bit reads; the values are handed
// out where they are used (lncc_lds.h).
template <int NV>
__device__ __forceinline__ void pairs_load(const float* __restrict__ src, lds_f2* q) {
#pragma unroll
    for (int m = 0; m < NV / 2; ++m) q[m] = reinterpret_cast<const lds_f2*>(src)[m];
}
template <int NV>
__device__ __forceinline__ void pairs_take(const lds_f2* q, float (&v)[NV]) {
    static_assert(NV % 2 == 0, "pairs");
#pragma unroll
    for (int m = 0; m < NV / 2; ++m) {
        lds_f2 f = q[m];
        asm("" : "+v"(f));
        v[2 * m] = f.x;
        v[2 * m + 1] = f.y;
    }
}

// Field q of (p, t, p^2, t^2, p t): its value, or a sum extended by it.
template <int Q>
__device__ __forceinline__ float field(float p, float t) {
    return Q == 0 ? p : Q == 1 ? t : Q == 2 ? p * p : Q == 3 ? t * t : p * t;
}
template <int Q>
__device__ __forceinline__ float field_add(float s, float p, float t) {
    return Q == 0 ? s + p : Q == 1 ? s + t : Q == 2 ? fmaf(p, p, s) : Q == 3 ? fmaf(t, t, s) : fmaf(p, t, s);
}

// The pieces of a launch, chunks of at most `most` planes of a tile: workgroup i takes pieces i,
// i + grid, ... in turn. The pieces of one chunk index lie side by side, so that the workgroups
// running at one time march through neighbouring tiles at the same plane and share their halo
// columns in the L2 (an even split of the planes over the grid, whose shares start at different
// planes, gained nothing by its even load: it fetches the halos again).
struct Pieces {
    uint32_t i, n, tiles, chunks;
    int D, most;
    __device__ __forceinline__ Pieces(const FusedArgs& a)
        : n(a.npieces), tiles((uint32_t)(a.ntx * a.nty)), chunks((uint32_t)a.nzc), D(a.dimD), most(a.dchunk) {
        // workgroups go to the 8 XCDs round-robin: XCD j takes the j-th contiguous range of a round's
        // pieces
        const uint32_t nb = gridDim.x, bid = blockIdx.x;
        const uint32_t xcd = bid % 8u, q8 = nb / 8u, r8 = nb % 8u;
        i = xcd * q8 + min(xcd, r8) + bid / 8u;
    }
    // tile (of all volumes) and planes [z0, z1) of the next piece
    __device__ __forceinline__ bool next(uint32_t& tile, int& z0, int& z1) {
        if (i >= n) return false;
        const uint32_t c = i / tiles;
        tile = (c / chunks) * tiles + i % tiles;
        z0 = (int)(c % chunks) * most;
        z1 = min(z0 + most, D);
        i += gridDim.x;
        return true;
    }
};

// Tile -> volume, first input column, first output row. With WHOLE the tile that reaches past a row's
// end starts up to NC - 1 columns earlier (not the first tile, which has none there), so that the last
// columns of a lane are a row's last ones and no lane's columns are cut; `skip` is that number, by which
// its own output columns start later.
// Bound of a tile with cut lanes: its loads, NC times as many of 4 bytes each, up to half as long again
// as the tiles beside it, for which a launch of one round waits. Loss at 160x192x224 k = 7 36.7 -> 25.2
// us, 96^3 k = 9 12.7 -> 10.0, (2,16,128^3) k = 7 187 -> 178; map at 160x192x224 k = 7 33 -> 29,
// (2,64,64^3) k = 7 152 -> 134; widths without cut lanes within 2%. bfloat16 loads one by one always.
template <class G, int NC, bool WHOLE>
__device__ __forceinline__ void tile_origin(const FusedArgs& a, uint32_t tile, int64_t& b, int& x0, int& y0, int& skip) {
    const uint32_t tx = tile % (uint32_t)a.ntx, t = tile / (uint32_t)a.ntx;
    x0 = (int)tx * G::ADV;
    skip = 0;
    if (WHOLE && tx > 0 && x0 + G::RW > a.dimW) skip = (NC - (a.dimW - x0) % NC) % NC;
    x0 -= skip;
    y0 = (int)(t % (uint32_t)a.nty) * G::OY;
    b = (int64_t)(t / (uint32_t)a.nty);
}

template <int HH, int NC, bool BF16, int MODE>
__global__ __launch_bounds__((FwdGeo<HH, NC>::LANES), 1) void lncc_forward_kernel(FusedArgs a) {
    using G = FwdGeo<HH, NC>;
    constexpr int K = 2 * HH + 1;
    constexpr int ELEM = BF16 ? 2 : 4;
    constexpr float VS = range_scale(K), NF = (float)(K * K * K);
    __shared__ __align__(16) float Xs[2 * G::BUF];
    __shared__ double red[G::NYW];

    const int tid = threadIdx.x;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid) >> 6;
    const int D = a.dimD, Hd = a.dimH, Wd = a.dimW;

    Pieces pieces(a);
    const int64_t HW = (int64_t)Hd * Wd;

    if (wave_id < G::NFW) {
        // ---------------- F waves ----------------
        int l, iy;
        float* const xs = Xs + fwd_f_lane<G>(tid, l, iy);
        int z0, z1;
        uint32_t tile;
        while (pieces.next(tile, z0, z1)) {
        int64_t b;
        int x0, y0, skip;
        tile_origin<G, NC, !BF16>(a, tile, b, x0, y0, skip);
        // F runs planes [tb, zend), whose windows are centred on [z0, z1), Y one step (PPB planes) later
        const int tb = z0 + HH, zend = z1 + HH, nsteps = fwd_steps<G>(z1 - z0);
        const int gy = y0 - HH + iy, gx = x0 + NC * l;
        const bool row_in = gy >= 0 && gy < Hd;
        const uint32_t plane_bytes = (uint32_t)(HW * ELEM);
        const uint32_t at = ((uint32_t)gy * (uint32_t)Wd + (uint32_t)gx) * ELEM;   // used only inside the volume
        const int inside = row_in ? Wd - gx : 0;
        // float32 rows are one wide load per lane and field, except in a row's only tile where its right
        // edge cuts a lane's columns and the load would read the next row's: `inside` of them one by one
        const bool wide = !BF16 && (x0 + G::RW <= Wd || (Wd - x0) % NC == 0);
        uint32_t voff[BF16 ? NC : 1];
        voff[0] = inside > 0 ? at : kOOB;
        if constexpr (BF16) {
#pragma unroll
            for (int j = 1; j < NC; ++j) voff[j] = j < inside ? at + j * ELEM : kOOB;
        }
        const uint64_t PB = (uint64_t)HW * ELEM;
        // the ring's planes before the first: tb - K + 1 ... (possibly below 0: zero-sized)
        const int64_t first = (b * D + tb - K + 1) * (int64_t)PB;
        uint64_t pa = (uint64_t)(uintptr_t)a.pred + first, ta = (uint64_t)(uintptr_t)a.target + first;
        float pn[2][NC], tn[2][NC];   // p, t of this plane and the next
        auto fetch = [&](int z, float (&p)[NC], float (&t)[NC]) __attribute__((always_inline)) {
            const uint32_t n = z >= 0 && z < min(D, zend) ? plane_bytes : 0u;
            const rsrc_words rp = words_at(pa, n), rt = words_at(ta, n);
            if (wide) {
                load_run<NC>(rp, voff[0], p);
                load_run<NC>(rt, voff[0], t);
            } else {
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    const uint32_t v = BF16 ? voff[BF16 ? j : 0] : j < inside ? at + j * ELEM : kOOB;
                    p[j] = load_elem<BF16>(rp, v);
                    t[j] = load_elem<BF16>(rt, v);
                }
            }
            pa += PB;
            ta += PB;
        };
        float pring[NC][K], tring[NC][K], fpre[NC][5], ch[NC][5];
        constexpr int M = HH + 1;
        constexpr bool CH = HH >= 2 && NC * (2 * K + 10) <= 80;
        // The march starts with a block: the k - 1 planes before its first one only enter windows, as
        // the previous block, and go straight into their ring slots.
#pragma unroll
        for (int r = 1; r < K; ++r) {
            float p[NC], t[NC];
            fetch(tb - K + r, p, t);
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                pring[j][r] = p[j];
                tring[j][r] = t[j];
            }
        }
        fetch(tb, pn[0], tn[0]);
        fetch(tb + 1, pn[1], tn[1]);
        // the chain (zstep5): the previous block's sums over slots M .. K-1
        auto form_chain = [&]() __attribute__((always_inline)) {
            static_for<0, 5>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value;
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    ch[j][q] = field<q>(pring[j][K - 1], tring[j][K - 1]);
#pragma unroll
                    for (int s = K - 2; s >= M; --s) ch[j][q] = field_add<q>(ch[j][q], pring[j][s], tring[j][s]);
                }
            });
        };
        if constexpr (CH) form_chain();
        // The march is unrolled by 2 k: the ring slot is the plane's position in its block of k, the
        // buffers alternate with its parity.
        uint32_t buf = G::F_BUF0;   // LDS offset of the buffer being written
        for (int base = tb; base < tb + nsteps * G::PPB; base += 2 * K) {
            static_for<0, 2 * K>([&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value, r = u % K, par = u % 2;
                const int zi = base + u;
                if (zi - u % G::PPB >= tb + nsteps * G::PPB) return;   // whole steps
                float (&p)[NC] = pn[par];
                float (&t)[NC] = tn[par];
                const bool out = zi < zend;   // not in the last step, which is Y's alone
                static_for<0, 5>([&](auto qc) __attribute__((always_inline)) {
                    constexpr int q = decltype(qc)::value;
                    float zs[NC];
#pragma unroll
                    for (int j = 0; j < NC; ++j) {
                        fpre[j][q] = r == 0 ? field<q>(p[j], t[j]) : field_add<q>(fpre[j][q], p[j], t[j]);
                        zs[j] = fpre[j][q];
                    }
                    if (out) {
#pragma unroll
                        for (int s = r + 1; s < (CH && r < M ? M : K); ++s)
#pragma unroll
                            for (int j = 0; j < NC; ++j) zs[j] = field_add<q>(zs[j], pring[j][s], tring[j][s]);
                        if constexpr (CH && r < M)
#pragma unroll
                            for (int j = 0; j < NC; ++j) zs[j] += ch[j][q];
                        float o[NC];
                        xsum_row<HH, NC>(zs, o);
#pragma unroll
                        for (int j = 0; j < NC; ++j) xs[buf + (u % G::PPB) * G::PLANE + q * G::XP + j * 16 * G::XS] = o[j];
                    }
                });
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    pring[j][r] = p[j];
                    tring[j][r] = t[j];
                }
                if constexpr (CH && r == K - 1) form_chain();
                fetch(zi + 2, p, t);
                if constexpr (u % G::PPB == G::PPB - 1) {
                    __syncthreads();
                    buf = fwd_other<G>(buf);
                }
            });
        }
        }
    } else {
        // ---------------- Y waves ----------------
        int seg, x;
        const float* const xs = Xs + fwd_y_lane<G>(tid - 64 * G::NFW, seg, x);
        float ndr = a.ndr;
        asm("" : "+v"(ndr));   // in a vector register: an addition with a scalar operand takes twice the cycles
        double loss_acc = 0.0;
        constexpr int NY = G::SY + 2 * HH;
        int z0, z1;
        uint32_t tile;
        while (pieces.next(tile, z0, z1)) {
        int64_t b;
        int x0, y0, skip;
        tile_origin<G, NC, !BF16>(a, tile, b, x0, y0, skip);
        const int nsteps = fwd_steps<G>(z1 - z0);
        const int gx = x0 + x, gy = y0 + seg * G::SY;
        // a column is this tile's if both neighbours' columns of its window were there, or are outside
        // the volume
        const bool col = gx < Wd && (x0 == 0 || x >= HH + skip) && (x < G::RW - HH || x0 + G::RW >= Wd);
        bool core[G::SY];
#pragma unroll
        for (int i = 0; i < G::SY; ++i) core[i] = col && gy + i < Hd;
        uint32_t buf = G::Y_BUF0;   // the buffer written one step ago
        for (int st = 0; st < nsteps; ++st) {
            // the planes that this step's sums are centred on: zc .. zc + PPB - 1
            const int zc = z0 + (st - 1) * G::PPB;
            if (st > 0) {
                const float* const row = xs + buf;
                lds_f2 rows[G::PPB][5][NY / 2];
#pragma unroll
                for (int e = 0; e < G::PPB; ++e)
#pragma unroll
                    for (int q = 0; q < 5; ++q) pairs_load<NY>(row + e * G::PLANE + q * G::XP, rows[e][q]);
#pragma unroll
                for (int e = 0; e < G::PPB; ++e) {
                    float S[5][G::SY];
#pragma unroll
                    for (int q = 0; q < 5; ++q) {
                        float v[NY];
                        pairs_take<NY>(rows[e][q], v);
                        box_sums<HH, G::SY>(v, S[q]);
                    }
                    const bool count = zc + e < z1;
                    float lsum = -0.f;
#pragma unroll
                    for (int i = 0; i < G::SY; ++i) {
                        const float Sp = S[0][i], St = S[1][i], Spp = S[2][i], Stt = S[3][i], Spt = S[4][i];
                        const float X = fmaf(-Sp, St, NF * Spt);
                        const float VP = fmaxf(fmaf(-Sp, Sp, NF * Spp), 0.f) + ndr;
                        const float VT = (fmaxf(fmaf(-St, St, NF * Stt), 0.f) + ndr) * VS;   // VT s
                        const float cr = X * __builtin_amdgcn_rcpf(VP * VT);                // c / s
                        const float ncc = (X * VS) * cr;
                        const float nccc = __builtin_elementwise_minimum(ncc, 1.0f);   // NaN stays NaN
                        if constexpr (MODE == MODE_MAPS) {
                            if (count && core[i]) {
                                const bool live = ncc < 1.0f;
                                const float uu = cr * VT;
                                const float w = fmaf(-Sp, uu, St);
                                const int64_t o = ((b * D + zc + e) * Hd + gy + i) * (int64_t)Wd + gx;
                                a.ncc_map[o] = nccc;
                                if (a.a_map) {
                                    a.a_map[o] = live ? (-2.f * VS) * (cr * w) : 0.f;
                                    a.b_map[o] = live ? (-NF * VS) * (cr * uu) : 0.f;
                                    a.c_map[o] = live ? (2.f * NF * VS) * cr : 0.f;
                                }
                            }
                        } else {
                            // a select: a window past the volume or the tile's own columns may be all zeros,
                            // whose ncc at smooth_dr = 0 is 0 * inf, and NaN times a zero mask stays NaN
                            // (against such a mask's fma 0.5%; at k = 3 3-5% on launches of one round: 15.9
                            // -> 16.7 us for 6 float32 volumes of 75x91x109)
                            lsum += core[i] ? nccc : 0.f;
                        }
                    }
                    if constexpr (MODE != MODE_MAPS)
                        if (count) loss_acc += (double)lsum;
                }
            }
            __syncthreads();
            buf = fwd_other<G>(buf);
        }
        }
        if constexpr (MODE != MODE_MAPS) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off, 64);
            if ((tid & 63) == 0) red[wave_id - G::NFW] = loss_acc;
        }
    }
    if constexpr (MODE == MODE_MAPS) return;
    __syncthreads();
    if (tid == 0) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < G::NYW; ++w) sum += red[w];
        a.partials[blockIdx.x] = sum;
        // the reduction reads the gradient plan's number of partials, which may be larger
        for (uint32_t i = gridDim.x + blockIdx.x; i < a.nparts; i += gridDim.x) a.partials[i] = 0.0;
    }
}

}  // namespace fl
