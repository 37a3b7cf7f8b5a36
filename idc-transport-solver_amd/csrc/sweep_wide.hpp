// Staggered sweep with one lane per coefficient (k_wide_ref, and k_diag_sweep_split with WIDE), the material path
// for sweeps that are bound by the chain of their steps rather than by the chip's throughput.
//
// Lane g of row r owns coefficient g = e + P*d of the row's cell (P = 2: 4 lanes a row; P = 3, 4: 16 lanes a row, of
// which P = 3 uses 9): row g of the element inverse in its registers, one source value, one right-hand side, one
// result.  A step is the two traces from LDS, two multiply-adds for the right-hand side, and the product with the
// row's right-hand sides, which for P = 3 and 4 takes one instruction per term: the multiply-add reads its factor from
// a lane of its 16-lane row (row_newbcast).  A wave issues about 55 instructions a step where the lane-split sweep
// issues 200, for a quarter of the rows.  A cell's run is read and written by one instruction, so no wave is needed
// for the stores.  The same operations in the same order as there: the same bits.
//
// Bands, records, item order, the wave stagger and the reference-layout inflow follow split_item; band inflow and
// outflow are the work of two further waves, so that the compute waves, which all wait for the slowest at each barrier,
// run the same few instructions in every row (inside the first wave it cost a third of a step).
//
// Measured on one band of Q2 (FP64): 0.18 us a step with 8 rows, 0.24 with 24, 0.37 with 56, where the lane-split
// sweep takes 0.5; without its loads and stores 0.16, 0.20 and 0.31: what is left is the wave's own chain (LDS, 14
// dependent FP64 operations, barrier) and, with many rows, the issue slots of a CU's four SIMDs.  Kernel times against
// the lane-split sweep's stand at the rule that picks one (wide_most_rows).
#pragma once

namespace tsw {

template <int P>
__host__ __device__ constexpr int wide_lanes() {
    return P == 2 ? 4 : 16;
}
// Threads of the largest workgroup, with the two waves for its inflow and outflow: 56 rows at degrees 2 and 3, 224 at 1.
constexpr int kWideThreads = 1024, kWideHelpers = 2;

template <typename T, int P>
struct WideLds {  // LDS carve-up in units of T
    static constexpr int N = P * P, PS = vround<T>(P);
    static constexpr int XS = P * PS + (P * PS * (int)sizeof(T) % 128 == 0 ? Vec16<T>::W : 0);  // row stride of the cells
    // stride of the inverse's rows: rows a multiple of 64 bytes apart would share a few banks
    static constexpr int RS = vround<T>(N) + (vround<T>(N) * (int)sizeof(T) % 64 == 0 ? Vec16<T>::W : 0);
    size_t xs, inv, total;
    // [2][1 + slots][XS] solved cells, by step parity; row 0 holds the y-inflow traces of the band's first row, that of
    // x-degree d at d PS.  [M][N][RS] inverses
    __host__ __device__ WideLds(int slots, int M) {
        xs = 0;
        inv = xs + (size_t)2 * (slots + 1) * XS;
        total = inv + (size_t)M * N * RS;
    }
};

// sum_c A[c] * (b of lane c of the 16-lane row), in the order of c: fma(A[c], b_c, acc) from A[0] b_0.  The sum starts
// at -0, so the first multiply-add is the plain product, sign of zero included.  b may come straight from a VALU
// instruction, after which a DPP read waits two states (the s_nop).  Every lane of the wave must be active.
#define TSW_DPP(op, k) op "_dpp %0, %1, %" #k " row_newbcast:"
#define TSW_ROW " row_mask:0xf bank_mask:0xf\n\t"
#define TSW_DOT9(op)                                                                                                    \
    "s_nop 1\n\t" TSW_DPP(op, 2) "0" TSW_ROW TSW_DPP(op, 3) "1" TSW_ROW TSW_DPP(op, 4) "2" TSW_ROW TSW_DPP(op, 5) "3"     \
        TSW_ROW TSW_DPP(op, 6) "4" TSW_ROW TSW_DPP(op, 7) "5" TSW_ROW TSW_DPP(op, 8) "6" TSW_ROW TSW_DPP(op, 9) "7" TSW_ROW \
            TSW_DPP(op, 10) "8" TSW_ROW
#define TSW_DOT16(op)                                                                                                    \
    TSW_DOT9(op) TSW_DPP(op, 11) "9" TSW_ROW TSW_DPP(op, 12) "10" TSW_ROW TSW_DPP(op, 13) "11" TSW_ROW TSW_DPP(op, 14)       \
    "12" TSW_ROW TSW_DPP(op, 15) "13" TSW_ROW TSW_DPP(op, 16) "14" TSW_ROW TSW_DPP(op, 17) "15" TSW_ROW
template <typename T>
__device__ __forceinline__ T row_dot(const T (&A)[9], T b) {
    T acc = T(-0.0);
    if constexpr (sizeof(T) == 8)
        asm volatile(TSW_DOT9("v_fmac_f64") : "+&v"(acc) : "v"(b), "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(A[4]), "v"(A[5]),
            "v"(A[6]), "v"(A[7]), "v"(A[8]));
    else
        asm volatile(TSW_DOT9("v_fmac_f32") : "+&v"(acc) : "v"(b), "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(A[4]), "v"(A[5]),
            "v"(A[6]), "v"(A[7]), "v"(A[8]));
    return acc;
}
template <typename T>
__device__ __forceinline__ T row_dot(const T (&A)[16], T b) {
    T acc = T(-0.0);
    if constexpr (sizeof(T) == 8)
        asm volatile(TSW_DOT16("v_fmac_f64") : "+&v"(acc) : "v"(b), "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(A[4]), "v"(A[5]),
            "v"(A[6]), "v"(A[7]), "v"(A[8]), "v"(A[9]), "v"(A[10]), "v"(A[11]), "v"(A[12]), "v"(A[13]), "v"(A[14]), "v"(A[15]));
    else
        asm volatile(TSW_DOT16("v_fmac_f32") : "+&v"(acc) : "v"(b), "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(A[4]), "v"(A[5]),
            "v"(A[6]), "v"(A[7]), "v"(A[8]), "v"(A[9]), "v"(A[10]), "v"(A[11]), "v"(A[12]), "v"(A[13]), "v"(A[14]), "v"(A[15]));
    return acc;
}
template <typename T>
__device__ __forceinline__ T row_dot(const T (&A)[4], T b) {  // 4 lanes a row
    T acc = A[0] * group_bcast<4>(b, 0);
#pragma unroll
    for (int c = 1; c < 4; ++c) acc = fmadd(A[c], group_bcast<4>(b, c), acc);
    return acc;
}
#undef TSW_DOT16
#undef TSW_DOT9
#undef TSW_ROW
#undef TSW_DPP

// v[0..P) <- p[0..P), p 16-byte aligned
template <typename T, int P>
__device__ __forceinline__ void run_get(const T *p, T (&v)[P]) {
    if constexpr (P % Vec16<T>::W == 0) {
        lds_get<T, P>(p, v);
    } else {  // (no element past the run: it would cost registers and, once they are reused, a wait)
#pragma unroll
        for (int k = 0; k < P; ++k) v[k] = p[k];
    }
}

// One item: band wid / nq of ordinate wid % nq of the problem sp, by the whole workgroup (every thread calls it): the
// compute waves, then the feeder and the sender wave.
template <typename T, int P, int MODE, int D>
__device__ __forceinline__ void wide_item(const DiagSweepParams<T> &sp, unsigned wid) {
    constexpr int N = P * P, LG = wide_lanes<P>(), RPW = 64 / LG;  // rows per wavefront
    constexpr bool HASQ = (MODE & 1) != 0, HASPHI = (MODE & 2) != 0, REF = (MODE & 4) != 0;
    using Lds = WideLds<T, P>;
    constexpr int PS = Lds::PS, RS = Lds::RS, XS = Lds::XS;
    using U = typename ExchangeSentinel<T>::U;
    static_assert(!REF || MODE == 5, "reference-layout sweep: sources only");
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
    const int slots = ((int)blockDim.x - 64 * kWideHelpers) / LG;
    const Lds L(slots, sp.M);
    T *linv = lds + L.inv, *xs = lds + L.xs;
    const int side = (slots + 1) * XS;
    const DiagMap dm{nx, ny};
    const size_t ncell = (size_t)dm.cells();
    const int Q = q >= sp.qo3 ? 3 : (q >= sp.qo2 ? 2 : (q >= sp.qo1 ? 1 : 0));
    const int tid = threadIdx.x;
    const T xi = G(sp.xi)[q], eta = G(sp.eta)[q];
    const bool xneg = xi <= T(0), yneg = eta <= T(0);

    for (int k = tid; k < sp.M * N * N; k += blockDim.x) {  // dx dy A^{-1}
        const int m = k / (N * N), e = k - m * N * N, row = e / N, col = e - row * N;
        linv[((size_t)m * N + row) * RS + col] = G(sp.ainv)[((size_t)m * sp.nq + q) * N * N + e];
    }

    // Row rl solves column t - rl in the workgroup's step t, between barriers t and t + 1 of nbar + 1; wave w holds
    // row slots [w RPW, (w + 1) RPW) and works on the steps of its rows.
    const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6) * RPW;
    auto run_of = [&](int first) {
        const int n = nrows - first < RPW ? nrows - first : RPW;
        return n > 0 ? (n - 1 + nx + D - 1) / D * D : 0;
    };
    const int last0 = (nrows - 1) / RPW * RPW;
    int nbar = last0 + run_of(last0);
    if (last0 > 0 && last0 - RPW + run_of(last0 - RPW) > nbar) nbar = last0 - RPW + run_of(last0 - RPW);
    const unsigned long long ref_bytes = REF ? (unsigned long long)(nx + 2) * (ny + 2) * sp.nq * N * 8 : 0;
    const __amdgpu_buffer_rsrc_t rq = REF ? buf_rsrc(sp.qref, ref_bytes)
                                          : buf_rsrc(HASQ ? sp.qsrc + (size_t)q * N * ncell : nullptr,
                                                     HASQ ? (unsigned long long)N * ncell * sizeof(T) : 0);
    T sx = xneg ? T(-1) : T(1), sy = yneg ? T(-1) : T(1);
    asm volatile("" : "+v"(sx), "+v"(sy));
    auto y_trace = [&](const T (&c)[P]) {  // outflow y-trace of one x-degree: sum_b sy^b psi(d, b)
        T v = c[0];
#pragma unroll
        for (int b = 1; b < P; ++b) v = (b & 1) ? v + sy * c[b] : v + c[b];
        return v;
    };

    if (w0 >= slots) {
        // Two waves beside the compute waves, whose chain sets the pace and which so run the same few instructions in
        // every row.  Two, because a wait for a load also waits for the wave's earlier stores.
        const int lane = tid & 63, yd = (lane & 3) < P ? (lane & 3) : P - 1, yc = lane >> 2;
        const bool has_in = band > 0, has_out = band < nb - 1;
        const gptr<U> xout = G(reinterpret_cast<U *>(sp.xtr)) + ((size_t)q * (nb - 1) + band) * nx * P;
        const gptr<U> xin = xout - (size_t)nx * P;
        if (w0 >= slots + RPW) {
            // The sender: in step t the record of the last row's cell of step t - 1, and the record that the feeder
            // consumed in step t - 1 (column t's) emptied.
            auto send = [&](int t) {
                const int c = t - nrows;
                if (has_out && c >= 0 && c < nx && lane < P) {
                    T v[P];
                    run_get<T, P>(xs + ((t - 1) & 1) * side + nrows * XS + lane * PS, v);
                    xstore(xout + (size_t)c * P + lane, to_bits(y_trace(v)));
                }
                if (has_in && t < nx && lane < P) xstore(xin + (size_t)t * P + lane, ExchangeSentinel<T>::bits);
            };
            lds_barrier();
            for (int t = 0; t < nbar; ++t) {
                send(t);
                lds_barrier();
            }
            send(nbar);
            return;
        }
        // The feeder: column t + 1's y-inflow of the band's first row into LDS during step t.  Lane l holds x-degree l % 4
        // of the next column that is l / 4 modulo 16, from the records of the band below, the halo traces, or (reference
        // layout) the halo cells.  A load goes out every 4 steps and is looked at 7 steps later (with loads of 16 columns
        // at once, looked at 3 steps later, Q2 128 x 128 took 108 us instead of 91: about 1 us from another CU's store to
        // its value here held the step up), so a band some 14 columns behind
        // its upstream one never waits.
        const gptr<const U> yin = has_in ? gptr<const U>(xin) : G(reinterpret_cast<const U *>(sp.tin_y)) + (size_t)q * nx * P;
        const bool halo = REF && !has_in, none = !REF && !has_in && sp.tin_y == nullptr;
        int mine = yc;  // this lane's column
        bool have = false;
        U cur = 0, raw[2] = {0, 0};
        double yr[2][P];
        int from[2] = {-1, -1};  // the column that buffer b was loaded from
        auto load = [&](int b) {  // (columns past the mesh: the last one, not used)
            from[b] = mine;
            const int c = mine < nx ? mine : nx - 1;
            if (halo) {
                const int i = xneg ? nx - c : c + 1, j = yneg ? ny + 1 : 0;
                ref_run_ld<P>(rq, (unsigned)((((long long)i * (ny + 2) + j) * sp.nq + q) * N * 8) + 8u * (unsigned)(yd * P), yr[b]);
            } else if (!none) {
                raw[b] = xload<U>(yin + (size_t)c * P + yd);
            }
        };
        auto look = [&](int b) {  // takes what a load brought, if a value was missing
            if (halo) {
                double v = yr[b][0];
#pragma unroll
                for (int k = 1; k < P; ++k) v += (yneg && (k & 1)) ? -yr[b][k] : yr[b][k];
                raw[b] = to_bits(T(v));
            }
            // (a load that was under way when the lane moved on to another column is dropped)
            const bool ok = !have && from[b] == mine && (!has_in || raw[b] != ExchangeSentinel<T>::bits);
            cur = ok ? raw[b] : cur;
            have = have || ok;
        };
        auto put = [&](int c) {
            if (c >= nx) return;
            const bool now = yc == (c & 15);
            for (int it = 0; __ballot(now && !have) != 0; ++it) {
                if (it >= kSpinLimit || ((it & 255) == 255 && xload<int>(G(sp.abort_flag)) != 0)) {
                    if (it >= kSpinLimit) xstore<int>(G(sp.abort_flag), 1);
                    cur = have ? cur : 0;  // given up: the call reports it
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                load(0);
                look(0);
            }
            if (now) {
                if ((lane & 3) < P) xs[((c + 1) & 1) * side + yd * PS] = from_bits<T>(cur);
                have = false;
                mine += 16;
            }
        };
        load(0);
        look(0);
        put(0);
        lds_barrier();
        for (int t0 = 0; t0 < nbar; t0 += 8) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (t0 + k >= nbar) break;
                if (k == 0) load(0);
                if (k == 4) load(1);
                if (k == 7) look(0);
                if (k == 3 && t0 > 0) look(1);
                put(t0 + k + 1);
                lds_barrier();
            }
        }
        return;
    }

    const int nrun = run_of(w0);
    const int rw = (tid & 63) / LG, g = tid % LG < N ? tid % LG : N - 1, d = g / P, e = g % P;
    const int rl = w0 + rw;
    const bool row_ok = rl < nrows;
    const int r = R0 + (row_ok ? rl : nrows - 1);  // slots past the band's rows load its last row and store nothing
    const int ra = row_ok ? rw : (1 << 30);        // column at the wave's step t is t - ra
    T tx;  // x-trace of y-degree e: the inflow, then the outflow of the row's last cell
    if constexpr (REF) {
        const gptr<const double> h = G(sp.qref) + (((size_t)(xneg ? nx + 1 : 0) * (ny + 2) + (yneg ? ny - r : r + 1)) * sp.nq + q) * N + e;
        double s = h[0];
#pragma unroll
        for (int a = 1; a < P; ++a) s += (xneg && (a & 1)) ? -h[P * a] : h[P * a];
        tx = T(s);
    } else {
        tx = (row_ok && sp.tin_x) ? G(sp.tin_x)[((size_t)q * ny + r) * P + e] : T(0);
    }

    // Global addresses.  Diagonal layout: lane offset (row, plane) plus the diagonal's; off(s) + r stays inside the array
    // on every diagonal, whatever the row.  Reference layout: offsets of the lane's value (and of the cell's material)
    // of the column of the next fetch and of the last step, modulo 2^32: outside the mesh they read some other value of
    // the buffer, or zero past its end, that is not used.  Stores of rows without a cell go past the end of the
    // buffer, where they are dropped.
    const unsigned plane = (unsigned)(ncell * sizeof(T));
    const unsigned long long nplanes = (unsigned long long)N * ncell * sizeof(T);  // bytes of one ordinate
    const unsigned nowhere = REF ? (unsigned)ref_bytes : (unsigned)nplanes;
    const __amdgpu_buffer_rsrc_t rout = REF ? buf_rsrc(sp.psi_ref, ref_bytes) : buf_rsrc(sp.psi + (size_t)q * N * ncell, nplanes);
    const __amdgpu_buffer_rsrc_t rphi = buf_rsrc(HASPHI ? sp.phi + (size_t)Q * N * ncell : nullptr, HASPHI ? nplanes : 0);
    const __amdgpu_buffer_rsrc_t rsigs = buf_rsrc(HASPHI ? sp.sig_s + (size_t)Q * ncell : nullptr, HASPHI ? plane : 0);
    const __amdgpu_buffer_rsrc_t rmat = REF ? buf_rsrc(sp.mat_cell, (unsigned long long)(nx + 2) * (ny + 2) * 4)
                                            : buf_rsrc(sp.mat + (size_t)Q * ncell, ncell * 4);
    const unsigned vrow0 = (unsigned)r * (unsigned)sizeof(T), vrow = vrow0 + (unsigned)g * plane, vmat = (unsigned)r * 4u;
    const unsigned dstep = REF ? (unsigned)((xneg ? -1LL : 1LL) * (ny + 2) * sp.nq * N * 8) : 0;  // one column on
    const unsigned mstep = xneg ? 0u - 4u * (unsigned)(ny + 2) : 4u * (unsigned)(ny + 2);
    unsigned foff = REF ? ref_off(0, r, nx, ny, sp.nq, q, N, xneg, yneg) + 8u * (unsigned)g - (unsigned)ra * dstep : 0;
    unsigned moff = 4u * (unsigned)((xneg ? nx : 1) * (ny + 2) + (yneg ? ny - r : r + 1)) - (unsigned)ra * mstep;
    unsigned soff = foff - dstep;
    const int s_last = nx + ny - 2;
    DiagWalk fw{R0 + w0, (int)(dm.base(R0 + w0) - dm.rlo(R0 + w0))};  // diagonal of the next fetch
    int so[D];  // the diagonals of the ring's slots, as offsets
#pragma unroll
    for (int u = 0; u < D; ++u) so[u] = 0;

    PQ pq[D];
    T pf[D], ps[D];
    int pm[D];
    auto fetch = [&](int u) {
        if constexpr (REF) {
            pq[u] = buf_ld<double>(rq, foff, 0);
            pm[u] = buf_ld<int>(rmat, moff, 0);
            foff += dstep;
            moff += mstep;
        } else {
            so[u] = fw.off;
            const unsigned bo = (unsigned)fw.off * (unsigned)sizeof(T);
            if (HASQ) pq[u] = buf_ld<T>(rq, vrow, bo);
            if (HASPHI) {
                pf[u] = buf_ld<T>(rphi, vrow, bo);
                ps[u] = buf_ld<T>(rsigs, vrow0, bo);
            }
            pm[u] = buf_ld<int>(rmat, vmat, (unsigned)fw.off * 4u);
            if (fw.s < s_last) fw.next(nx, ny);
        }
    };

    T Arow[N];  // row g of the current material's dx dy A^{-1}
    int cur_mat = -1;
    const T kx = T((double)xi * (double)(xneg ? T(-(2 * d + 1)) : T(((d & 1) ? -1 : 1) * (2 * d + 1))) / (double)sp.dx);
    const T ky = T((double)eta * (double)(yneg ? T(-(2 * e + 1)) : T(((e & 1) ? -1 : 1) * (2 * e + 1))) / (double)sp.dy);
    const T *ysr = xs + (size_t)rl * XS + d * PS;        // the row below's cell: its coefficients of x-degree d
    const T *xsr = xs + (size_t)(rl + 1) * XS + e;       // this row's: its coefficients of y-degree e
    T *xsw = xs + (size_t)(rl + 1) * XS + d * PS + e;    // (lanes without a coefficient repeat that of lane N - 1)
    const bool row0 = rl == 0;
    T xo = T(0);  // this lane's coefficient of the last solved cell
    bool act = false;  // the last step solved a cell in this lane's row
    auto store_last = [&](int off) {
        if constexpr (REF) {
            buf_st<double>(rout, act ? soff : nowhere, 0, (double)xo);
            soff += dstep;
        } else {
            buf_st<T>(rout, act ? vrow : nowhere, (unsigned)off * (unsigned)sizeof(T), xo);
        }
    };

    if (nrun > 0) {
#pragma unroll
        for (int u = 0; u < D - 1; ++u) fetch(u);
    }
    for (int k = 0; k <= w0 && k <= nbar; ++k) lds_barrier();  // the first one publishes the inverse table
    int col = -ra;
    for (int t0 = 0; t0 < nrun; t0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int pr = D % 2 == 0 ? (u + 1) & 1 : (t0 + u + 1) & 1;  // LDS side of the last step
            T yv[P], xv[P];
            run_get<T, P>(ysr + pr * side, yv);
#pragma unroll
            for (int a = 0; a < P; ++a) xv[a] = xsr[pr * side + a * PS];
            __builtin_amdgcn_sched_barrier(0);
            store_last(so[(u + D - 1) % D]);
            fetch((u + D - 1) % D);
            __builtin_amdgcn_sched_barrier(0);
            const bool now = (unsigned)col < (unsigned)nx;
            if (pm[u] != cur_mat && now) {
                cur_mat = pm[u];
                lds_get<T, N>(linv + ((size_t)cur_mat * N + g) * RS, Arow);
            }
            T a;
            if (HASPHI) {
                const T wsc = T(1) * ps[u] * T(kInv4Pi);
                a = HASQ ? fmadd(wsc, pf[u], T(pq[u])) : wsc * pf[u];
            } else {
                a = T(pq[u]);
            }
            T v = xv[0];  // outflow x-trace: sum_a sx^a psi(a, e)
#pragma unroll
            for (int i = 1; i < P; ++i) v = (i & 1) ? v + sx * xv[i] : v + xv[i];
            tx = act ? v : tx;
            T ty = y_trace(yv);
            ty = row0 ? yv[0] : ty;
            act = now;
            ++col;
            xo = row_dot(Arow, fmadd(ky, ty, fmadd(kx, tx, a)));
            xsw[(1 - pr) * side] = xo;
            lds_barrier();
        }
    }
    if (nrun > 0) store_last(so[D - 1]);
    for (int k = w0 + nrun; k < nbar; ++k) lds_barrier();
}

}  // namespace tsw
