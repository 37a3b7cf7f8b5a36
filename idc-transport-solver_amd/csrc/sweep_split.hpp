// Lane-split staggered sweep (k_diag_sweep_split, k_split_ref), the material path with LG lanes per mesh row:
// LG = 2 for P = 2 and 4 for P = 3, 4 (for P = 3 the fourth lane repeats the third and stores nothing).
//
// Lane g of row r owns the coefficients k = e + P*g (e < P) of the row's cell.  At a step it loads the sources of
// its coefficients, forms their right-hand sides from the row's x-trace and its own y-trace value, broadcasts them
// to the row's other lanes with DPP quad permutations, applies its P rows of the element inverse to the whole
// right-hand side and leaves its coefficients in LDS, from which the row's lanes form the x-trace of the next step
// and the row above its y-trace.  A band of 64 rows fills four wavefronts at degrees 2 and 3, so an ordinate's sweep
// spreads over four times as many SIMDs as with a lane per row.  Every value is computed by the same operations, in
// the same order, as the material path of k_diag_sweep (sums of products are written as explicit fused multiply-adds
// in both), so the two kernels give the same bits.
//
// Bands and exchange records follow k_diag_sweep; the band's first and last rows consume and fill the records
// themselves, as its one-wave variant does.  A wave works only on the steps at which one of its rows has a cell.
//
// MODE bit 4 (with bit 1, sources only): the source is read from `qref` and psi written to `psi_ref`, both in the
// reference layout [i][j][q][d][e], and the inflow is read from the halo cells of qref, so no layout conversion and
// no launch for the traces is needed.  Lane g's coefficients are one contiguous run of P doubles there, and the LG
// lanes of a row cover the cell's run.  Two further waves (kSplitStorers) write the results, or, where more workgroups
// on a CU or more rows in one pay more, the lanes themselves (which of the two: storers_forced and the rules after it).
// BATCH: the workgroup's parameters are batch[items[b].x], and items[b].y = band * nq + ordinate, numbered band-major
// so that a band's upstream band is always dispatched first; items with a negative problem index are padding.
//
// What bounds the reference layout (Q2 S12 on 280 x 280, 561 steps a workgroup, FP64, kernel time): not HBM, which
// would take 190 us, nor the arithmetic of the chain of steps (290 us with the loads and stores taken out), but the
// memory instructions' way through the address unit and the L1 between a step's barriers: each takes 16 cycles
// whatever its width, a load of 16 rows' 72-byte runs about 50 from the L2, and a store about 5 cycles per 64-byte
// segment that it touches.  Against 527 us for stores by the compute lanes (each segment in two or three pieces) and
// items in plain order:
//   - one L2 sees the whole cache lines of neighbouring ordinates (take_item): less HBM traffic, and loads from the
//     L2 instead of behind it;
//   - stores as whole runs, read back from LDS by two storer waves a step later: 472 us; by the compute lanes
//     themselves 489 us, by one storer wave 514 us;
//   - the x-trace from LDS instead of 18 DPP moves, no address arithmetic in the step, idle waves only at barriers.
// Two or four ordinates side by side in a workgroup (whole lines per access, shorter bands) took 490 to 530 us, all
// memory instructions in two memory waves 706 us.  Other kernels, before and after: Q1 280 x 280 250 -> 215 us; Q2
// 32 x 32 53 -> 39, 128 x 128 172 -> 145; Q3 32 x 32 97 -> 61, 128 x 128 270 -> 223, 256 x 256 667 -> 461 us.
#pragma once

namespace tsw {

// Lanes per row of the lane-split sweep for DG order P (P rows of the element inverse per lane).
template <int P>
__host__ __device__ constexpr int split_lanes() {
    return P == 2 ? 2 : 4;
}
// The lane-split sweep keeps a lane's P rows of the inverse in registers: built where they fit
// (Q1-Q3 in both precisions; an FP64 Q3 lane holds 64 doubles, about 230 VGPRs in all, two waves per SIMD).
template <typename T, int P>
__host__ __device__ constexpr bool split_supported() {
    return P >= 2 && P <= 4 && P * P * P * (int)sizeof(T) <= 64 * 8;
}

// REF: reference layout; CELLS: with storer waves
template <typename T, int P, bool REF, bool CELLS>
struct SplitLds {  // LDS carve-up in units of T, 16-byte aligned arrays and rows
    static constexpr int N = P * P;
    static constexpr int PS = vround<T>(P), RS = vround<T>(P * N);
    // row stride of the solved cells: P runs of PS values, and a 16-byte pad where P runs are a multiple of
    // 128 bytes, so that a wave's rows do not all start in one LDS bank
    static constexpr int XS = P * PS + (P * PS * (int)sizeof(T) % 128 == 0 ? Vec16<T>::W : 0);
    static constexpr int YR = 64 / split_lanes<P>();  // columns of the y-inflow ring: the rows of a wave
    size_t ex, xs, lin, inv, total;
    // slots: row slots of the workgroup; M: materials ([M][P][RS] inverse rows, lane g's block at g).  With
    // storer waves the solved cells of two steps are kept ([2][slots][XS]): the rows above take their
    // y-traces, and the storers the results, from the last step's
    __host__ __device__ SplitLds(int slots, int M) {
        ex = 0;                                                 // [slots][2][PS] y-traces between rows, by step parity
        xs = ex + (CELLS ? 0 : (size_t)2 * slots * PS);         // [slots][XS] solved cells, for the rows' x-traces
        lin = xs + (size_t)(CELLS ? 2 : 1) * slots * XS;        // [YR][PS] y-inflow traces of row 0 (reference layout)
        inv = lin + (REF ? (size_t)YR * PS : 0);                // [M][P][RS]
        total = inv + (size_t)M * P * RS;
    }
};
// Most row slots of a workgroup of 512 threads with `storers` storer waves.
template <int P>
__host__ __device__ constexpr int split_max_slots(int storers) {
    return (512 - 64 * storers) / split_lanes<P>();
}

// v read from lane K of its LG-lane group (quad permutation; K is a constant after unrolling)
template <int LG>
__device__ __forceinline__ int group_bcast_i(int v, int K) {
    if constexpr (LG == 4) {
        switch (K) {
            case 0: return __builtin_amdgcn_mov_dpp(v, 0x00, 0xf, 0xf, false);
            case 1: return __builtin_amdgcn_mov_dpp(v, 0x55, 0xf, 0xf, false);
            case 2: return __builtin_amdgcn_mov_dpp(v, 0xAA, 0xf, 0xf, false);
            default: return __builtin_amdgcn_mov_dpp(v, 0xFF, 0xf, 0xf, false);
        }
    } else {  // pairs: lanes (0,1) read lane K, lanes (2,3) read lane 2+K
        switch (K) {
            case 0: return __builtin_amdgcn_mov_dpp(v, 0xA0, 0xf, 0xf, false);
            default: return __builtin_amdgcn_mov_dpp(v, 0xF5, 0xf, 0xf, false);
        }
    }
}
template <int LG, typename T>
__device__ __forceinline__ T group_bcast(T v, int K) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, group_bcast_i<LG>(__builtin_bit_cast(int, v), K));
    } else {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        const unsigned lo = (unsigned)group_bcast_i<LG>((int)(unsigned)b, K);
        const unsigned hi = (unsigned)group_bcast_i<LG>((int)(unsigned)(b >> 32), K);
        return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
    }
}

// P contiguous doubles of a reference-layout run at byte offset off: 16-byte accesses, then an 8-byte one
// for odd P (off is a multiple of 8; buffer accesses of several dwords need only dword alignment)
template <int P>
__device__ __forceinline__ void ref_run_ld(__amdgpu_buffer_rsrc_t r, unsigned off, double (&v)[P]) {
    typedef unsigned V4 __attribute__((ext_vector_type(4)));
    typedef unsigned V2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < P / 2; ++i) {
        const V4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 16 * i, 0);
        v[2 * i] = __builtin_bit_cast(double, V2{x[0], x[1]});
        v[2 * i + 1] = __builtin_bit_cast(double, V2{x[2], x[3]});
    }
    if constexpr (P % 2 != 0) v[P - 1] = buf_ld<double>(r, off, 8 * (P - 1));
}
// v (as doubles) to P contiguous doubles at byte offset off, in the same pieces as ref_run_ld
template <typename T, int P>
__device__ __forceinline__ void ref_run_st(__amdgpu_buffer_rsrc_t r, unsigned off, const T (&v)[P]) {
    typedef unsigned V4 __attribute__((ext_vector_type(4)));
    typedef unsigned V2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < P / 2; ++i) {
        const V2 a = __builtin_bit_cast(V2, (double)v[2 * i]), b = __builtin_bit_cast(V2, (double)v[2 * i + 1]);
        __builtin_amdgcn_raw_buffer_store_b128(V4{a[0], a[1], b[0], b[1]}, r, (int)off, 16 * i, 0);
    }
    if constexpr (P % 2 != 0) buf_st<double>(r, off, 8 * (P - 1), (double)v[P - 1]);
}

// Waits until the exchange record value *rec (already loaded once into v) is filled; on the spin limit, or
// when another band has given up (*abort_flag), returns zero and the caller proceeds.
template <typename T>
__device__ __forceinline__ typename ExchangeSentinel<T>::U wait_value(gptr<const typename ExchangeSentinel<T>::U> rec,
                                                                      typename ExchangeSentinel<T>::U v,
                                                                      gptr<int> abort_flag) {
    using U = typename ExchangeSentinel<T>::U;
#pragma unroll 1
    for (int it = 0; v == ExchangeSentinel<T>::bits; ++it) {
        if (it >= kSpinLimit || ((it & 255) == 255 && xload<int>(abort_flag) != 0)) {
            if (it >= kSpinLimit) xstore<int>(abort_flag, 1);
            return 0;
        }
        __builtin_amdgcn_s_sleep(1);
        v = xload<U>(rec);
    }
    return v;
}

// One item of the lane-split sweep: band wid / nq of ordinate wid % nq of the problem sp, by the whole
// workgroup (every thread calls it; it ends with a workgroup barrier).  ST: its storer waves (reference layout).
template <typename T, int P, int MODE, int D, int ST>
__device__ __forceinline__ void split_item(const DiagSweepParams<T> &sp, unsigned wid) {
    constexpr int N = P * P, LG = split_lanes<P>(), RPW = 64 / LG;  // rows per wavefront
    constexpr bool HASQ = (MODE & 1) != 0, HASPHI = (MODE & 2) != 0, REF = (MODE & 4) != 0, CELLS = ST > 0;
    using Lds = SplitLds<T, P, REF, CELLS>;
    constexpr int PS = Lds::PS, RS = Lds::RS, XS = Lds::XS;
    using U = typename ExchangeSentinel<T>::U;
    static_assert(REF ? MODE == 5 : ST == 0, "reference-layout lane-split sweep: sources only; storers there alone");
    using PQ = typename std::conditional<REF, double, T>::type;  // prefetched source (converted at use)
    const int nb = sp.nbands < 2 ? 1 : sp.nbands;
    const int q = (int)(wid % (unsigned)sp.nq);
    const int band = (int)(wid / (unsigned)sp.nq);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *lds = reinterpret_cast<T *>(smem_raw);
    const int nx = sp.nx, ny = sp.ny;
    const int BR = nb > 1 ? sp.band_rows : ny;
    const int R0 = band * BR;
    const int nrows = BR < ny - R0 ? BR : ny - R0;
    const int slots = ((int)blockDim.x - 64 * ST) / LG;
    const Lds L(slots, sp.M);
    T *linv = lds + L.inv;
    const DiagMap dm{nx, ny};
    const size_t ncell = (size_t)dm.cells();
    const int Q = q >= sp.qo3 ? 3 : (q >= sp.qo2 ? 2 : (q >= sp.qo1 ? 1 : 0));
    const int tid = threadIdx.x;
    const T xi = G(sp.xi)[q], eta = G(sp.eta)[q];
    const bool xneg = xi <= T(0), yneg = eta <= T(0);

    // the table holds dx dy A^{-1}, row-blocked so lane g's P rows are one aligned LDS run
    for (int k = tid; k < sp.M * N * N; k += blockDim.x) {
        const int m = k / (N * N), e = k - m * N * N, row = e / N, col = e - row * N;
        linv[((size_t)m * P + row / P) * RS + (row % P) * N + col] = G(sp.ainv)[((size_t)m * sp.nq + q) * N * N + e];
    }

    // Wave w holds row slots [w RPW, (w + 1) RPW) and works on its own steps t = 0 .. live_n - 1 (row rw of the
    // wave solves column t - rw), starting w RPW barriers after the workgroup's first step; every wave passes
    // nbar barriers in all.
    const int rw = (tid & 63) / LG, g = tid % LG;
    const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6) * RPW;  // first row slot of this wave
    auto run_of = [&](int first) {  // steps of the wave at row `first`, rounded up to whole rings
        const int n = nrows - first < RPW ? nrows - first : RPW;
        return n > 0 ? (n - 1 + nx + D - 1) / D * D : 0;
    };
    const int last0 = (nrows - 1) / RPW * RPW;
    int nbar = last0 + run_of(last0);
    if (last0 > 0 && last0 - RPW + run_of(last0 - RPW) > nbar) nbar = last0 - RPW + run_of(last0 - RPW);
    const int nrun = run_of(w0);
    const unsigned long long ref_bytes = REF ? (unsigned long long)(nx + 2) * (ny + 2) * sp.nq * N * 8 : 0;
    const unsigned dstep = REF ? (unsigned)((xneg ? -1LL : 1LL) * (ny + 2) * sp.nq * N * 8) : 0;  // one column on
    // stores of lanes without a cell go to this offset, past the end of the buffer, where they are dropped: a
    // store then always issues, and the waits for the loads behind it count it (behind a branch it might not,
    // and each wait would also cover the loads of one or two later steps)
    const unsigned long long nplanes = (unsigned long long)N * ncell * sizeof(T);  // bytes of one ordinate
    const unsigned nowhere = REF ? (unsigned)ref_bytes : (unsigned)nplanes;
    const __amdgpu_buffer_rsrc_t rout = REF ? buf_rsrc(sp.psi_ref, ref_bytes) : buf_rsrc(sp.psi + (size_t)q * N * ncell, nplanes);

    if constexpr (ST > 0) if (w0 >= slots) {
        // The storer waves: step t's cells during step t + 1, from LDS, as the band's runs one after the other
        // (access m of lane l, m dealt round the storers, is values (l + 64 m) SW of them).  A 64-byte segment of L2
        // takes a write request of its own, about one in 4 cycles per CU: written by the compute lanes, a cell's run
        // goes out in pieces, each segment in two requests or more, and the compute waves wait for the queue.
        constexpr int SW = P % 2 == 0 ? 2 : 1, SM = (split_max_slots<P>(ST) * N / SW + 64 * ST - 1) / (64 * ST);
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));  // (keeps these tables out of the compute waves' registers)
        const int m0 = __builtin_amdgcn_readfirstlane((tid >> 6) - slots * LG / 64);
        unsigned soff[SM];   // byte offset of step t's cell
        int c0[SM], at[SM];  // its column is t - c0 (far outside the mesh past the band's rows), its LDS offset
#pragma unroll
        for (int m = 0; m < SM; ++m) {
            const int e = (lane + 64 * (m * ST + m0)) * SW, row = e / N, k = e - row * N;
            const bool ok = row < nrows;
            c0[m] = ok ? row : (1 << 30);
            at[m] = ok ? row * XS + k / P * PS + k % P : 0;
            soff[m] = ref_off(0, R0 + (ok ? row : 0), nx, ny, sp.nq, q, N, xneg, yneg) + 8u * (unsigned)k - (unsigned)c0[m] * dstep;
        }
        lds_barrier();
        for (int t = 0; t < nbar; ++t) {
            lds_barrier();
            const T *xt = lds + L.xs + (t & 1) * slots * XS;
            T v[SM][SW];
#pragma unroll
            for (int m = 0; m < SM; ++m)
#pragma unroll
                for (int k = 0; k < SW; ++k) v[m][k] = xt[at[m] + k];
#pragma unroll
            for (int m = 0; m < SM; ++m) {
                if (64 * (m * ST + m0) * SW < nrows * N)  // wave-uniform
                    ref_run_st<T, SW>(rout, (unsigned)(t - c0[m]) < (unsigned)nx ? soff[m] : nowhere, v[m]);
                soff[m] += dstep;
            }
        }
        return;
    }

    const int rl = w0 + rw;
    const int dd = g < P ? g : P - 1;  // the x-degree whose coefficients this lane owns
    const bool owner = g < P;
    const bool row_ok = rl < nrows;
    const int rc = row_ok ? rl : nrows - 1;  // slots past the band's rows load its last row and store nothing
    const int r = R0 + rc;
    const int ra = row_ok ? rw : (1 << 30);  // column at step t is t - ra: never inside the mesh without a row
    T tx;  // x-trace of y-degree dd: the inflow, then the outflow of the row's last cell
    if constexpr (REF) {
        const gptr<const double> h = G(sp.qref) + (((size_t)(xneg ? nx + 1 : 0) * (ny + 2) + (yneg ? ny - r : r + 1)) * sp.nq + q) * N + dd;
        double s = h[0];
#pragma unroll
        for (int a = 1; a < P; ++a) s += (xneg && (a & 1)) ? -h[P * a] : h[P * a];
        tx = T(s);
    } else {
        tx = (row_ok && sp.tin_x) ? G(sp.tin_x)[((size_t)q * ny + r) * P + dd] : T(0);
    }

    // global addresses.  Diagonal layout: lane offset (row, first plane) plus a scalar offset (diagonal,
    // plane); off(s) + r stays inside the array on every diagonal s of the mesh, whatever the row.
    // Reference layout: the lane's byte offset of its run, moved by one column a step while inside the mesh.
    const unsigned plane = (unsigned)(ncell * sizeof(T));
    const unsigned dplane = (unsigned)(dd * P) * plane;  // byte offset of this lane's first plane (< N * plane)
    const __amdgpu_buffer_rsrc_t rq = REF ? buf_rsrc(sp.qref, ref_bytes)
                                          : buf_rsrc(HASQ ? sp.qsrc + (size_t)q * N * ncell : nullptr, HASQ ? nplanes : 0);
    const __amdgpu_buffer_rsrc_t rphi = buf_rsrc(HASPHI ? sp.phi + (size_t)Q * N * ncell : nullptr, HASPHI ? nplanes : 0);
    const __amdgpu_buffer_rsrc_t rsigs = buf_rsrc(HASPHI ? sp.sig_s + (size_t)Q * ncell : nullptr, HASPHI ? plane : 0);
    const __amdgpu_buffer_rsrc_t rmat = buf_rsrc(sp.mat + (size_t)Q * ncell, ncell * 4);
    const unsigned dref = 8u * (unsigned)(dd * P);  // byte offset of this lane's run within a cell's run
    const unsigned vrow0 = (unsigned)r * (unsigned)sizeof(T), vrow = vrow0 + dplane;
    const unsigned vmat = (unsigned)r * 4u;
    unsigned foff = REF ? ref_off(0, r, nx, ny, sp.nq, q, N, xneg, yneg) + dref : 0;  // run of the next fetch
    unsigned soff = foff;  // (no storers) run of the row's next result
    const int s_last = nx + ny - 2;
    DiagWalk fw{R0 + w0, (int)(dm.base(R0 + w0) - dm.rlo(R0 + w0))};  // diagonal of the next fetch
    DiagWalk cw{fw.s - 1, fw.s > 0 ? (int)(dm.base(fw.s - 1) - dm.rlo(fw.s - 1)) : 0};  // diagonal of the last step
    // exchange records: read from the band below (xin), written for the band above (xout)
    const gptr<U> xtr = G(reinterpret_cast<U *>(sp.xtr)) + ((size_t)q * (nb - 1) + band) * nx * P;
    const bool has_in = band > 0, has_out = band < nb - 1;
    const gptr<U> xin = xtr - (size_t)nx * P, xout = xtr;
    // y-inflow of the band's first row, column by column: the records of the band below, or the halo traces
    // (the reference layout takes the latter from the halo cells themselves, through the LDS ring `lin`)
    const gptr<const U> yin = has_in ? gptr<const U>(xin) : G(reinterpret_cast<const U *>(sp.tin_y)) + (size_t)q * nx * P;
    const bool first = w0 == 0, ywave = first && (has_in || (!REF && sp.tin_y != nullptr));
    const bool xrow = has_in && rl == 0;  // consumes the records of the band below
    // reference layout, band 0: lane (rw, g) of the first wave loads the run of column c0 + rw's y-inflow halo
    // cell, RPW columns ahead of their use
    const bool yhalo = REF && first && band == 0;
    double yr[REF ? P : 1];
    auto yfetch = [&](int c0) {
        if constexpr (REF) {
            const int c = c0 + rw < nx ? c0 + rw : nx - 1, i = xneg ? nx - c : c + 1, j = yneg ? ny + 1 : 0;
            ref_run_ld<P>(rq, (unsigned)((((long long)i * (ny + 2) + j) * sp.nq + q) * N * 8) + dref, yr);
        }
    };
    const bool lastrow = has_out && owner && rl == nrows - 1;

    PQ pq[D][HASQ ? P : 1];
    T pf[D][HASPHI ? P : 1], ps[D];
    int pm[D];
    U px[D];
    int ft = 0;
    auto fetch = [&](int u) {
        const unsigned so = (unsigned)fw.off * (unsigned)sizeof(T), sm = (unsigned)fw.off * 4u;
        if constexpr (REF) {
            ref_run_ld<P>(rq, foff, pq[u]);
            foff += (unsigned)(ft - ra) < (unsigned)(nx - 1) ? dstep : 0u;
        } else if (HASQ) {
#pragma unroll
            for (int e = 0; e < P; ++e) pq[u][e] = buf_ld<T>(rq, vrow, so + e * plane);
        }
        if (HASPHI) {
#pragma unroll
            for (int e = 0; e < P; ++e) pf[u][e] = buf_ld<T>(rphi, vrow, so + e * plane);
            ps[u] = buf_ld<T>(rsigs, vrow0, so);
        }
        pm[u] = buf_ld<int>(rmat, vmat, sm);
        if (ywave && ft < nx) px[u] = xload<U>(yin + (size_t)ft * P + dd);
        if (fw.s < s_last) fw.next(nx, ny);
        ++ft;
    };

    T Arow[P * N];  // rows dd*P .. dd*P + P-1 of the current material's dx dy A^{-1}
    int cur_mat = -1;
    T kxo, kye[P];  // face couplings divided by dx dy (rounded once), this lane's x-degree for kx
    {
        const T kd = xneg ? T(-(2 * dd + 1)) : T(ipow_m1(dd) * (2 * dd + 1));
        kxo = T((double)xi * (double)kd / (double)sp.dx);
#pragma unroll
        for (int e = 0; e < P; ++e) {
            const T ke = yneg ? T(-(2 * e + 1)) : T(ipow_m1(e) * (2 * e + 1));
            kye[e] = T((double)eta * (double)ke / (double)sp.dy);
        }
    }
    T sx = xneg ? T(-1) : T(1), sy = yneg ? T(-1) : T(1);
    asm volatile("" : "+v"(sx), "+v"(sy));
    // LDS: the row below's y-trace or, with storer waves, its cell's coefficients of this lane's x-degree, and the
    // row's own cell, of the last step; where this step's go
    const int side = CELLS ? slots * XS : PS;  // between the two steps' copies
    const int sb = rl > 0 ? rl - 1 : 0;  // the row below
    const T *exr = CELLS ? lds + L.xs + (size_t)sb * XS + dd * PS : lds + L.ex + (size_t)sb * 2 * PS + dd;
    T *exw = lds + L.ex + (size_t)rl * 2 * PS + dd;
    const T *xsr = lds + L.xs + (size_t)rl * XS + dd;
    T *xsw = lds + L.xs + (size_t)rl * XS + dd * PS;
    auto y_trace = [&](const T (&c)[P]) {  // outflow y-trace of one x-degree: sum_b sy^b psi(d, b)
        T v = c[0];
#pragma unroll
        for (int b = 1; b < P; ++b) v = (b & 1) ? v + sy * c[b] : v + c[b];
        return v;
    };
    T *lin = lds + L.lin + dd;
    T xo[P];  // this lane's coefficients of the last solved cell
#pragma unroll
    for (int e = 0; e < P; ++e) xo[e] = T(0);
    bool act = false;  // the last step solved a cell in this lane's row

    // results of the last step to memory (diagonal layout: cw stands at its diagonal)
    auto store_last = [&]() {
        if constexpr (REF && ST == 0) {
            ref_run_st<T, P>(rout, act && owner ? soff : nowhere, xo);
            soff += act ? dstep : 0u;
        } else if constexpr (!REF) {
            const unsigned so = (unsigned)cw.off * (unsigned)sizeof(T), vo = act && owner ? vrow : nowhere;
#pragma unroll
            for (int e = 0; e < P; ++e) buf_st<T>(rout, vo, so + e * plane, xo[e]);
            if (cw.s < s_last) cw.next(nx, ny);
        }
    };

    if (nrun > 0) {
        if (yhalo) yfetch(0);
#pragma unroll
        for (int u = 0; u < D - 1; ++u) fetch(u);
    }
    for (int k = 0; k <= w0 && k <= nbar; ++k) lds_barrier();  // the first one publishes the inverse table
    for (int t0 = 0; t0 < nrun; t0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int t = t0 + u;
            const int pr = D % 2 == 0 ? (u + 1) & 1 : (t + 1) & 1;  // LDS side of the last step
            // the traces the cell needs come through LDS; meanwhile the last step's cell goes out and the ring
            // slot it freed is refilled
            T yv[P], xv[P];
            if constexpr (CELLS) lds_get<T, P>(exr + pr * side, yv);
            else yv[0] = exr[pr * side];
#pragma unroll
            for (int d = 0; d < P; ++d) xv[d] = xsr[(CELLS ? pr * side : 0) + d * PS];
            __builtin_amdgcn_sched_barrier(0);
            store_last();
            fetch((u + D - 1) % D);
            __builtin_amdgcn_sched_barrier(0);
            T v = xv[0];  // outflow x-trace: sum_a sx^a psi(a, dd)
#pragma unroll
            for (int a = 1; a < P; ++a) v = (a & 1) ? v + sx * xv[a] : v + xv[a];
            tx = act ? v : tx;
            T ty = CELLS ? y_trace(yv) : yv[0];
            act = (unsigned)(t - ra) < (unsigned)nx;
            if (pm[u] != cur_mat && act) {
                cur_mat = pm[u];
                lds_get<T, P * N>(linv + ((size_t)cur_mat * P + dd) * RS, Arow);
            }
            if (first) {
                U y = 0;
                if (REF && yhalo) {
                    if (t % RPW == 0) {  // the next RPW columns' traces
                        double s = yr[0];
#pragma unroll
                        for (int b = 1; b < (REF ? P : 1); ++b) s += (yneg && (b & 1)) ? -yr[b] : yr[b];
                        lin[rw * PS] = T(s);
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                        yfetch(t + RPW);
                    }
                    y = to_bits(lin[t % RPW * PS]);
                } else if (ywave) {
                    if (xrow && act) {
                        px[u] = wait_value<T>(xin + (size_t)t * P + dd, px[u], G(sp.abort_flag));
                        if (owner) xstore(xin + (size_t)t * P + dd, ExchangeSentinel<T>::bits);
                    }
                    y = px[u];
                }
                ty = rl == 0 ? (act ? from_bits<T>(y) : T(0)) : ty;
            }
            T Bo[P];  // right-hand side of coefficients e + P dd
#pragma unroll
            for (int e = 0; e < P; ++e) {
                T a;
                if (HASPHI) {
                    const T wsc = T(1) * ps[u] * T(kInv4Pi);
                    a = HASQ ? fmadd(wsc, pf[u][e], T(pq[u][e])) : wsc * pf[u][e];
                } else {
                    a = T(pq[u][e]);
                }
                Bo[e] = fmadd(kye[e], ty, fmadd(kxo, group_bcast<LG>(tx, e), a));
            }
            T B[N];
#pragma unroll
            for (int d = 0; d < P; ++d)
#pragma unroll
                for (int e = 0; e < P; ++e) B[e + P * d] = group_bcast<LG>(Bo[e], d);
#pragma unroll
            for (int e = 0; e < P; ++e) {
                T acc = Arow[e * N] * B[0];
#pragma unroll
                for (int col = 1; col < N; ++col) acc = fmadd(Arow[e * N + col], B[col], acc);
                xo[e] = acc;
            }
            if constexpr (!CELLS) exw[(1 - pr) * side] = y_trace(xo);
            lds_put<T, P>(xsw + (CELLS ? (1 - pr) * side : 0), xo);
            if (lastrow && act) xstore(xout + (size_t)(t - ra) * P + dd, to_bits(y_trace(xo)));
            lds_barrier();
        }
    }
    if (nrun > 0) store_last();
    for (int k = w0 + nrun; k < nbar; ++k) lds_barrier();
}

}  // namespace tsw

#include "sweep_wide.hpp"

namespace tsw {

// Work counters of a persistent launch: two sets of one counter per XCD, each in a cache line of its own;
// a launch takes items with one set and clears the other for the next launch.  Batch launches add the item
// range of each XCD's queue.
constexpr int kWorkStride = 16, kWorkSet = kXcds * kWorkStride, kWorkTable = kSplitWorkTable;
static_assert(kWorkTable == 2 * kWorkSet, "two sets of counters before the table");

// The next item of a persistent launch as {queue, position}, or position -1 when every queue is empty; by the
// whole workgroup.  A workgroup drains its own XCD's queue first, then the others'.  Items with neighbouring
// ordinates, whose cell runs share cache lines in the reference layout, are in one queue: one L2 then sees the
// whole lines, where workgroups of several XCDs would each fetch them and write parts of them.  Items of a queue
// are taken in order, so a band's upstream band, which is in the same queue before it, has always been taken by a
// running workgroup.
template <typename Len>
__device__ __forceinline__ int2 take_item(int *work, Len len) {
    __shared__ int2 next;
    if (threadIdx.x < 64) {
        const int lane = (int)threadIdx.x;
        const int own = __builtin_amdgcn_s_getreg((3 << 11) | 20) & (kXcds - 1);  // XCC_ID
        int pick = own, pos = -1;
        for (;;) {  // leaves when an item is taken or every counter is past its queue's end
            int k = 0;
            if (lane == 0) k = atomicAdd(work + pick * kWorkStride, 1);
            k = __builtin_amdgcn_readfirstlane(k);
            if (k < len(pick)) {
                pos = k;
                break;
            }
            const bool more = lane < kXcds && xload<int>(G(work) + lane * kWorkStride) < len(lane);
            const unsigned m = (unsigned)__ballot(more) & ((1u << kXcds) - 1);
            if (m == 0) break;
            pick = (own + __builtin_ctz((m >> own | m << (kXcds - own)) & ((1u << kXcds) - 1))) & (kXcds - 1);
        }
        if (lane == 0) next = int2{pick, pos};
    }
    __syncthreads();
    const int2 k{__builtin_amdgcn_readfirstlane(next.x), __builtin_amdgcn_readfirstlane(next.y)};
    __syncthreads();  // every thread has read `next` before it is written again
    return k;
}

// One problem (sp1, workgroup = band x ordinate), a batch with one item per workgroup (items[b] = {problem,
// band * nq + ordinate}, a negative problem marking padding), or a persistent batch launch (work != null,
// counter set `set`): items ordered by queue, work[kWorkTable + x] the first item of XCD x's queue.
template <typename T, int P, int MODE, int D, bool BATCH, bool WIDE, int ST>
__global__ __launch_bounds__(WIDE ? kWideThreads : 512) void k_diag_sweep_split(DiagSweepParams<T> sp1, const DiagSweepParams<T> *__restrict__ batch,
                                                          const int2 *__restrict__ items, int *__restrict__ work, int set) {
    if constexpr (!BATCH) {
        if (sp1.skip && *G(sp1.skip)) return;  // a replayed iteration after the loop has stopped
        if constexpr (WIDE) wide_item<T, P, MODE, D>(sp1, blockIdx.x);
        else split_item<T, P, MODE, D, ST>(sp1, blockIdx.x);
    } else {
        if (work && blockIdx.x == 0 && threadIdx.x < kXcds) work[(1 - set) * kWorkSet + threadIdx.x * kWorkStride] = 0;
        const gptr<const int> table = G(static_cast<const int *>(work)) + kWorkTable;
        size_t at = blockIdx.x;
        do {
            if (work) {
                const int2 k = take_item(work + set * kWorkSet, [&](int x) { return table[x + 1] - table[x]; });
                if (k.y < 0) break;  // workgroup-uniform: every wave leaves
                at = (size_t)(table[k.x] + k.y);
            }
            const gptr<const int> it = G(reinterpret_cast<const int *>(items)) + 2 * at;
            const int item_p = it[0], item_v = it[1];
            if (item_p < 0) continue;  // padding of an XCD-ordered item list
            const DiagSweepParams<T> sp = batch[item_p];
            if (sp.skip && *G(sp.skip)) continue;
            split_item<T, P, MODE, D, ST>(sp, (unsigned)item_v);
        } while (work);
    }
}

// Items (source, ordinate, band) of the sweeps of n right-hand sides src.psi[r] of one problem in place on the reference
// layout: the (source, ordinate) pairs split evenly into the XCDs' queues, each queue band-major.
struct RefItems {
    int pairs, nb;
    __device__ RefItems(const int n, const int nq, const int nbands) : pairs(n * nq), nb(nbands < 2 ? 1 : nbands) {}
    __device__ int first(int x) const { return x * pairs / kXcds; }  // first pair of queue x
    __device__ int count(int x) const { return (first(x + 1) - first(x)) * nb; }
};
// Makes sp the problem of position pos of queue x and returns its item number (band * nq + ordinate).
template <typename T, int P>
__device__ __forceinline__ unsigned ref_item(DiagSweepParams<T> &sp, const SplitSources &src, const RefItems &I, int x, int pos, T *xtr) {
    const int p0 = I.first(x), np = I.first(x + 1) - p0, pair = p0 + pos % np, band = pos / np, r = pair / sp.nq;
    sp.qref = src.psi[r];
    sp.psi_ref = src.psi[r];
    sp.xtr = xtr + (size_t)r * sp.nq * (I.nb - 1) * sp.nx * P;  // the source's exchange records
    return (unsigned)(band * sp.nq + pair - r * sp.nq);
}

// One workgroup per item (work null: workgroup b takes item b / 8 of queue b % 8, the XCD that it is sent to), or a
// persistent launch taking items.  The launch does nothing while *changed == mark.
template <typename T, int P, int D, int ST>
__global__ __launch_bounds__(512) void k_split_ref(DiagSweepParams<T> sp, SplitSources src, int n, int *__restrict__ work, int set,
                                                   const int *__restrict__ changed, int mark) {
    T *const xtr = sp.xtr;
    const RefItems I(n, sp.nq, sp.nbands);
    if (work && blockIdx.x == 0 && threadIdx.x < kXcds) work[(1 - set) * kWorkSet + threadIdx.x * kWorkStride] = 0;
    if (changed && *G(changed) == mark) return;  // the inputs are not those the tables were built from
    int2 k{(int)(blockIdx.x % kXcds), (int)(blockIdx.x / kXcds)};
    do {
        if (work) k = take_item(work + set * kWorkSet, [&](int x) { return I.count(x); });
        if (k.y < 0 || k.y >= I.count(k.x)) break;  // workgroup-uniform: every wave leaves
        split_item<T, P, 5, D, ST>(sp, ref_item<T, P>(sp, src, I, k.x, k.y, xtr));
    } while (work);
}

// The same with a lane per coefficient and one workgroup per item: the loop of a persistent launch costs 40 registers,
// and with them a third of the waves on a CU; the queue's atomics cost 2 us of a call.
template <typename T, int P, int D>
__global__ __launch_bounds__(kWideThreads) void k_wide_ref(DiagSweepParams<T> sp, SplitSources src, int n,
                                                           const int *__restrict__ changed, int mark) {
    const RefItems I(n, sp.nq, sp.nbands);
    if (changed && *G(changed) == mark) return;
    const int x = (int)(blockIdx.x % kXcds), pos = (int)(blockIdx.x / kXcds);
    if (pos >= I.count(x)) return;  // past the end of a shorter queue
    wide_item<T, P, 5, D>(sp, ref_item<T, P>(sp, src, I, x, pos, sp.xtr));
}

}  // namespace tsw
