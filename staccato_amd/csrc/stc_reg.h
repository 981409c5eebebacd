// stc_reg.h -- register-resident solve of small systems (gfx950), n <= 128.
//
// The whole matrix of a point lives in the registers of one workgroup: lane l
// of every wavefront holds rows l + 64 t (t < RM), and blocks of four columns are
// dealt to the wavefronts in turn (CPW columns each).  A block's owner finds its
// pivots (one DPP maximum and a ballot per column) and publishes the multipliers
// through LDS; after one barrier every wavefront reads the pivot rows' entries of
// its own columns by v_readlane and applies the rank-4 update.  Rows never move;
// lpos[t] is a row's LAPACK position.
//
// What bounds it: the issue slots of the updates (a readlane pair per pivot and
// column, four FMAs per row) and one latency chain per column (pivot search and
// reciprocal); there is no memory traffic inside.  The
// unblocked LDS factorisation that this replaces read and wrote every trailing
// entry through LDS and took two barriers per column; the 16-column register
// panel for n = 65..128 sent the trailing matrix through the caches per panel.
//
//   complex128 (plain): P A = L U with zgetrf's pivots; right-hand sides are
//     extra columns, so their forward elimination is free.  U goes to LDS packed
//     by columns (n (n + 1) / 2 entries) as its columns finish, and each
//     wavefront substitutes back for its own right-hand sides without a
//     barrier.  The adjoint reuses the region for L packed by rows.
//   complex64 (refined): the inverse by Gauss-Jordan elimination with the same
//     pivots, in place: it costs the rank-1 updates of the finished rows and
//     columns (idle lanes and registers otherwise), and every solve of the
//     refinement becomes one product with a register-resident matrix instead
//     of two triangular solves.  The FP64 residual decides convergence, as with
//     LU factors (same number of steps: 2.0 on average to 1e-15, either way).
#pragma once

namespace stc {

// ---- wavefront maxima ------------------------------------------------------------------------
// maximum of non-negative doubles (NaN counts as the largest, so it propagates)
__device__ __forceinline__ double wave_dmax(double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v) & 0x7FFFFFFFFFFFFFFFull;
    wave_argmax64(b);
    return __longlong_as_double((long long)b);
}
// max |z| over the wavefront's rows (NaN propagates); the squares decide
// unless they leave the range of a double
template <int RM>
__device__ __forceinline__ double wave_zmax(const z64 (&z)[RM]) {
    double q = 0.0;
#pragma unroll
    for (int t = 0; t < RM; ++t) q = nmax(q, fma(z[t].re, z[t].re, z[t].im * z[t].im));
    const double m = wave_dmax(q);
    if ((m > 1e-290 && m < 1e300)) return sqrt(m);
    double h = 0.0;
#pragma unroll
    for (int t = 0; t < RM; ++t) h = nmax(h, zabs(z[t]));
    return wave_dmax(h);
}

// ---- pivot search of one column (its wavefront) ----------------------------------------------------
// First row in LAPACK order of the largest |re| + |im| among rows with
// lpos >= jj (izamax's NaN rule, pivot_ukey).  The high words of the keys are
// reduced; only ties look at the low words and then at the positions.
template <typename T, int RM>
__device__ __forceinline__ void reg_pivot(const cx<T> (&col)[RM], const int (&lpos)[RM], int jj, int& pln, int& tw) {
    unsigned hi[RM], m = 0;
    unsigned long long key[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        key[t] = lpos[t] >= jj ? pivot_ukey(cabs1(col[t]), lpos[t] == jj) : 0ull;
        hi[t] = sizeof(T) == 4 ? (unsigned)key[t] : (unsigned)(key[t] >> 32);
        // complex128: eligible rows stay above the others whose high word is 0
        if (sizeof(T) == 8) hi[t] = lpos[t] >= jj ? hi[t] + 1u : 0u;
        m = hi[t] > m ? hi[t] : m;
    }
    m = wave_umax(m);
    auto tied = [&](auto&& is, int& cnt) {
        cnt = 0;
#pragma unroll
        for (int t = 0; t < RM; ++t) {
            const unsigned long long b = __ballot(is(t));
            if (b) {
                tw = t;
                pln = __builtin_ctzll(b);
            }
            cnt += __popcll(b);
        }
    };
    int cnt;
    tied([&](int t) { return hi[t] == m; }, cnt);
    if (cnt == 1) return;
    unsigned ml = 0;
    if (sizeof(T) == 8) {
#pragma unroll
        for (int t = 0; t < RM; ++t) {
            const unsigned v = hi[t] == m ? (unsigned)key[t] : 0u;
            ml = v > ml ? v : ml;
        }
        ml = wave_umax(ml);
    }
    auto in = [&](int t) { return hi[t] == m && (sizeof(T) == 4 || (unsigned)key[t] == ml); };
    unsigned mp = 0;
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        const unsigned v = in(t) ? (unsigned)(1024 - lpos[t]) : 0u;
        mp = v > mp ? v : mp;
    }
    mp = wave_umax(mp);
    tied([&](int t) { return in(t) && (unsigned)(1024 - lpos[t]) == mp; }, cnt);
}

// Fast form of the search: the high words of |re| + |im| alone (complex64: the whole
// word).  True when one row has the largest and its magnitude is far from both
// ends of the range, so that neither ties, zeros, infinities and NaN nor a
// scaled reciprocal have to be thought of (reg_pivot and crecip do that).
template <typename T, int RM>
__device__ __forceinline__ bool reg_pivot_fast(const cx<T> (&col)[RM], const int (&lpos)[RM], int jj, int& pw) {
    unsigned hi[RM], m = 0;
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        const T v = cabs1(col[t]);
        unsigned h;
        if constexpr (sizeof(T) == 4) h = __float_as_uint(v);
        else h = (unsigned)__double2hiint(v);
        hi[t] = lpos[t] >= jj ? h : 0u;
        m = hi[t] > m ? hi[t] : m;
    }
    m = wave_umax(m);
    // 2^-60 .. 2^60 (complex64), 2^-500 .. 2^500
    constexpr unsigned kLo = sizeof(T) == 4 ? (127u - 60u) << 23 : (1023u - 500u) << 20;
    constexpr unsigned kHi = sizeof(T) == 4 ? (127u + 60u) << 23 : (1023u + 500u) << 20;
    int cnt = 0, pln = 0, tw = 0;
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        const unsigned long long b = __ballot(hi[t] == m);
        if (RM == 1) {
            pln = __builtin_ctzll(b | (1ull << 63));
        } else if (b) {
            tw = t;
            pln = __builtin_ctzll(b);
        }
        cnt += __popcll(b);
    }
    pw = pln | (tw << 6);
    return cnt == 1 && m - kLo < kHi - kLo;
}
// 1 / z for z in that range
__device__ __forceinline__ cx<float> recip_mid(cx<float> z) {
    const float r = __builtin_amdgcn_rcpf(fmaf(z.re, z.re, z.im * z.im));
    return cmk<float>(z.re * r, -z.im * r);
}
__device__ __forceinline__ z64 recip_mid(z64 z) {
    const double q = fma(z.re, z.re, z.im * z.im);
    double r = __builtin_amdgcn_rcp(q);
    r = fma(fma(-q, r, 1.0), r, r);
    r = fma(fma(-q, r, 1.0), r, r);
    return cmk<double>(z.re * r, -z.im * r);
}

// LDS of one point's elimination
template <typename T>
struct RegLds {
    cx<T>* lcol;  // two (DEFER: three) alternating sets of four multiplier columns (n each)
    int* pos;     // the rows' positions, handed from owner to owner
    int* sc;      // [4 set + j]: pivot lane | slot << 6 of a block's columns; [12]: first zero pivot (1-based) or 0
    cx<T>* rp;    // reciprocals of the pivots, by column
    cx<T>* U;     // LU: U packed by columns
};

// Column of register column i (block columns of four, dealt to the wavefronts in
// turn; rot: blocks this wavefront has finished, each moved to the back)
template <int NW, int CPW>
__device__ __forceinline__ int reg_col(int i, int rot, int wave) {
    int slot = (i >> 2) + rot;
    slot = slot >= CPW / 4 ? slot - CPW / 4 : slot;
    return 4 * (NW * slot + wave) + (i & 3);
}

// ---- elimination ------------------------------------------------------------------------------
// x: the matrix (see the top of the file); b: NE extra columns per wavefront, ne of
// them in use.  GJ: Gauss-Jordan with unscaled pivot rows (row p of the result
// is multiplied by the reciprocal of its pivot where it is used): column jj
// becomes -multipliers, 1 in the pivot row.  Otherwise LU: U's columns go to R.U
// and, with KEEPL, the negated multipliers stay in the rows below.  R.rp: the
// reciprocals of the pivots, by column.
//
// Blocks of four columns belong to one wavefront, which factors them without a
// barrier; the others meet the block's four pivots in one rank-4 update (the
// pivot row's entry of step k is read after the updates of steps < k).  The
// owner of the next block only updates and factors that block while the others
// are still updating; with DEFER its other columns get both blocks' updates one
// pass later, so a pass is as long as the factorisation of one block (measured:
// complex64 n <= 64 and complex128 n > 64 gain, 123 -> 104 us at n = 47, 1501 points; two
// workgroups of complex64 n > 64 are bound by issue slots and lose 6 %, and n = 60 in
// complex128 needs the LDS of the third multiplier set for a fourth workgroup).
// Blocks of four against one column per barrier: 175k -> 148k cycles a point at
// n = 60 (complex128).  A wavefront's next block is always x[0..3]
// (finished blocks rotate to the back), so every register index is static and
// the loop has one body.  Returns the wavefront's rotation (see reg_col).
template <typename T, int NW, int RM, int CPW, int NE, bool GJ, bool DEFER, bool KEEPL>
__device__ __forceinline__ int reg_eliminate(cx<T> (&x)[CPW][RM], cx<T> (&b)[NE ? NE : 1][RM], int ne,
                                             int (&lpos)[RM], int n, const RegLds<T>& R) {
    constexpr int NS = CPW / 4;
    static_assert(CPW % 4 == 0 && NS >= 2, "blocks of four columns");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = (n + 3) >> 2;
    // entry of the pivot row (lane pw & 63, slot pw >> 6) in a column, uniform
    auto pivot_entry = [&](const cx<T> (&c)[RM], int pw) {
        cx<T> u = c[0];
#pragma unroll
        for (int t = 1; t < RM; ++t) {
            u.re = (pw >> 6) == t ? c[t].re : u.re;
            u.im = (pw >> 6) == t ? c[t].im : u.im;
        }
        return cbcast(u, pw & 63);
    };
    // factors x[0..3] = columns 4 blk ..; publishes the negated multipliers and the pivots
    auto factor_block = [&](int blk, int set) {
        cx<T>* lb = R.lcol + set * 4 * n;
        int pws[4];
        cx<T> rps[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int jj = 4 * blk + j;
            pws[j] = 0;
            rps[j] = czero<T>();
            if (jj >= n) {  // last block: no such column, zero multipliers
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (lane + 64 * t < n) stc<3>(lb + (j * n + 64 * t + lane), czero<T>());
                continue;
            }
            int pw;
            cx<T> rp;
            if (reg_pivot_fast<T, RM>(x[j], lpos, jj, pw)) {
                rp = recip_mid(pivot_entry(x[j], pw));
            } else {
                int pln = 0, tw = 0;
                reg_pivot<T, RM>(x[j], lpos, jj, pln, tw);
                pw = pln | (tw << 6);
                const cx<T> pv = pivot_entry(x[j], pw);
                const bool zero = pv.re == T(0) && pv.im == T(0);
                rp = crecip(pv);
                rp.re = zero ? T(0) : rp.re;
                rp.im = zero ? T(0) : rp.im;
                if (zero && lane == 0 && lds1<3>(R.sc + 12) == 0) stc1i(R.sc + 12, jj + 1);
            }
            pws[j] = pw;
            rps[j] = rp;
            const int pln = pw & 63, tw = pw >> 6;
            int bpos = lpos[0];
#pragma unroll
            for (int t = 1; t < RM; ++t) bpos = tw == t ? lpos[t] : bpos;
            bpos = __builtin_amdgcn_readlane(bpos, pln);
            cx<T> l[RM];
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const bool piv = lane == pln && tw == t;
                const bool sub = GJ ? !piv : (!piv && lpos[t] >= jj);
                l[t] = cmul(x[j][t], cmk<T>(-rp.re, -rp.im));
                l[t].re = sub ? l[t].re : T(0);
                l[t].im = sub ? l[t].im : T(0);
                if (lane + 64 * t < n) stc<3>(lb + (j * n + 64 * t + lane), l[t]);
                if (GJ) {
                    x[j][t].re = piv ? T(1) : l[t].re;
                    x[j][t].im = l[t].im;
                } else if (KEEPL) {
                    x[j][t].re = sub ? l[t].re : x[j][t].re;
                    x[j][t].im = sub ? l[t].im : x[j][t].im;
                }
                lpos[t] = piv ? jj : (lpos[t] == jj ? bpos : lpos[t]);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (GJ ? c != j : c > j) {
                    const cx<T> u = pivot_entry(x[c], pw);
#pragma unroll
                    for (int t = 0; t < RM; ++t) cfma(x[c][t], l[t], u);
                }
        }
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                stc1i(R.sc + 4 * set + j, pws[j]);
                if (4 * blk + j < n) stc<3>(R.rp + 4 * blk + j, rps[j]);
            }
        }
#pragma unroll
        for (int t = 0; t < RM; ++t)
            if (lane + 64 * t < n) stc1i(R.pos + (64 * t + lane), lpos[t]);
        // the finished block to the back
        cx<T> r[4][RM];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int t = 0; t < RM; ++t) r[u][t] = x[u][t];
#pragma unroll
        for (int i = 0; i + 4 < CPW; ++i)
#pragma unroll
            for (int t = 0; t < RM; ++t) x[i][t] = x[i + 4][t];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int t = 0; t < RM; ++t) x[CPW - 4 + u][t] = r[u][t];
    };
    // for each of a set's four pivots: f(pivot, its negated multipliers), the next
    // one's loaded ahead
    auto each_pivot = [&](int set, auto&& f) {
        const cx<T>* lb = R.lcol + set * 4 * n;
        cx<T> l[RM], ln[RM];
        int pw = lds1<3>(R.sc + 4 * set), pn = 0;
#pragma unroll
        for (int t = 0; t < RM; ++t) l[t] = ldc<3>(lb + min(64 * t + lane, n - 1));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int kn = min(k + 1, 3);
            pn = lds1<3>(R.sc + 4 * set + kn);
#pragma unroll
            for (int t = 0; t < RM; ++t) ln[t] = ldc<3>(lb + (kn * n + min(64 * t + lane, n - 1)));
            f(uniform(pw), l);
            pw = pn;
#pragma unroll
            for (int t = 0; t < RM; ++t) l[t] = ln[t];
        }
    };
    auto update = [&](cx<T> (&c)[RM], int pw, const cx<T> (&l)[RM]) {
        const cx<T> u = pivot_entry(c, pw);
#pragma unroll
        for (int t = 0; t < RM; ++t) cfma(c[t], l[t], u);
    };
    constexpr int NSET = DEFER ? 3 : 2;
    int rot = 0, set = NSET - 1;
    // one loop body for every block: pass -1 factors block 0 only
#pragma nounroll
    for (int blk = -1; blk < nb; ++blk) {
        const int nset = set == NSET - 1 ? 0 : set + 1;  // of block blk + 1
        const bool next = blk + 1 < nb && wave == (blk + 1) % NW;
        const bool mine = blk >= 0 && wave == blk % NW;
        if (next) {
            if (blk >= 0) {
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (lane + 64 * t < n) lpos[t] = lds1<3>(R.pos + (64 * t + lane));
                each_pivot(set, [&](int pw, const cx<T> (&l)[RM]) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) update(x[j], pw, l);
                });
            }
            factor_block(blk + 1, nset);
            ++rot;
        }
        if (!GJ && mine) {
            // U of the block factored in the previous pass (now the back group): rows whose
            // position is final and above (or at) the diagonal
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int jj = 4 * blk + j;
                if (jj < n)
#pragma unroll
                    for (int t = 0; t < RM; ++t)
                        if (lpos[t] >= 0 && lpos[t] <= jj)
                            stc<3>(R.U + (((jj * (jj + 1)) >> 1) + lpos[t]), x[CPW - 4 + j][t]);
            }
        }
        if (blk >= 0 && !(DEFER && next)) {
            // the wavefront's other columns; where its own block was factored in the previous
            // pass, they still miss the block before it (DEFER)
            int s0 = set;
            if (DEFER && mine && blk > 0) s0 = set == 0 ? 2 : set - 1;
            const bool back = GJ && (mine || next);  // the back group is that block (up to date)
#pragma nounroll
            for (;;) {
                each_pivot(s0, [&](int pw, const cx<T> (&l)[RM]) {
                    // opaque copies: conditions invariant in the loops would be unswitched
                    // out of them, a copy of the body each, and the code would outgrow the
                    // instruction cache
                    int nbl = nb, nel = ne;
                    asm volatile("" : "+s"(nbl), "+s"(nel));
#pragma unroll
                    for (int g = 0; g < NS; ++g) {
                        int slot = g + rot;
                        if (GJ) slot = slot >= NS ? slot - NS : slot;
                        // absent and (LU) finished blocks are left alone
                        if (slot < NS && NW * slot + wave < nbl && !(g == NS - 1 && back)) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) update(x[4 * g + j], pw, l);
                            // keeps the groups apart: the pivot-row entries of all columns
                            // at once would not fit the scalar registers
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < NE; ++e)
                        if (e < nel) update(b[e], pw, l);
                });
                if (s0 == set) break;
                s0 = set;
            }
        }
        set = nset;
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < RM; ++t)
        if (lane + 64 * t < n) lpos[t] = lds1<3>(R.pos + (64 * t + lane));
    return rot >= NS ? rot - NS : rot;
}

// The point's descriptor, loaded anew by each phase: kept over the elimination,
// its fields would take the scalar registers of the pivot rows.
__device__ __forceinline__ SysDesc reg_sys(const SysDesc* sp, int fidx) {
    unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)sp);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((uintptr_t)sp >> 32));
    asm volatile("" : "+s"(lo));  // not merged with the previous phase's loads
    SysDesc s = load_uniform(reinterpret_cast<const SysDesc*>(((uintptr_t)hi << 32) | lo));
    if (s.op_stride) {  // one explicit matrix per frequency index
        const long long o = (long long)fidx * s.op_stride;
        s.K += o;
        s.M += o;
        if (s.has_D) s.D += o;
    }
    if (s.f_stride) s.F += (long long)fidx * s.f_stride;
    return s;
}

// ---- results of a point that was not solved (info > 0) -----------------------------------------
__device__ __forceinline__ void reg_singular(const SysDesc& s, int fidx, int info, int nthreads) {
    const int tid = threadIdx.x;
    const double2 qn = make_double2(__builtin_nan(""), __builtin_nan(""));
    if (s.X) {
        double2* X = s.X + (size_t)fidx * s.ldx * s.nrhs;
        for (int e = tid; e < s.n * s.nrhs; e += nthreads) X[e % s.n + (size_t)(e / s.n) * s.ldx] = qn;
    }
    if (s.Y) {
        double2* Y = s.Y + (size_t)fidx * s.nout * s.nrhs;
        for (int e = tid; e < s.nout * s.nrhs; e += nthreads) Y[e] = qn;
    }
    if (s.berr)
        for (int g = tid; g < s.nrhs; g += nthreads) s.berr[(size_t)fidx * s.nrhs + g] = __builtin_inf();
    if (s.adj_out)
        for (int q = tid; q < s.p + 2; q += nthreads) s.adj_out[(size_t)fidx * (s.p + 2) + q] = 0.0;
    if (tid == 0) {
        s.info[fidx] = info;
        if (s.iters) s.iters[fidx] = 0;
    }
}

// ==== complex64 with FP64 refinement ==============================================================
// One point.  Wavefront g looks after right-hand side g of a group of four: its
// residual norms, scaling and solution are wavefront-local, and only the
// products with A and with its inverse (columns split over the wavefronts) meet
// in LDS: four barriers per refinement step.
template <int RM, int CPW>
__device__ __forceinline__ void reg_point_refined(const SysDesc* sp, int fidx, const KParams& kp, char* smem) {
    using C = cx<float>;
    constexpr int NW = 4, G = 4;
    const int n = __builtin_amdgcn_readfirstlane(sp->n), tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    RegLds<float> R;
    char* p = smem;
    R.lcol = reinterpret_cast<C*>(p);
    p += align16((RM == 1 ? 12LL : 8LL) * n * 8);
    R.pos = reinterpret_cast<int*>(p);
    p += align16(n * 4LL);
    R.sc = reinterpret_cast<int*>(p);
    p += 64;
    R.rp = reinterpret_cast<C*>(p);
    p += align16(n * 8LL);
    R.U = nullptr;
    double* ds = reinterpret_cast<double*>(p);  // [g]: backward error of column g
    p += align16(16 * 8);
    z64* xs = reinterpret_cast<z64*>(p);
    p += align16(4LL * n * 16);
    char* parts = p;
    p += align16(4LL * 4 * n * 16);
    C* rv = reinterpret_cast<C*>(p);  // [column][g]
    int row[RM];
    bool in[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        in[t] = lane + 64 * t < n;
        row[t] = in[t] ? lane + 64 * t : n - 1;
    }
    // ---- A(w) in FP64, its row sums, and the rounded copy in registers
    C x[CPW][RM];
    double asum[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) asum[t] = 0.0;
    {
        const SysDesc s = reg_sys(sp, fidx);
        const double w = s.freq ? kTwoPi * s.freq[fidx] : 0.0, w2 = w * w;
        with_kind(s, [&](auto kc) {
            constexpr int KIND = decltype(kc)::value;
            constexpr int QC = RM == 1 || KIND == kOpOne ? 4 : 2;
#pragma unroll
            for (int qc = 0; qc < CPW; qc += QC) {
                z64 a[QC][RM];
                const bool any = reg_col<NW, CPW>(qc & ~3, 0, 0) < n;
                if (any) {
#pragma unroll
                    for (int q = 0; q < QC; ++q)
#pragma unroll
                        for (int t = 0; t < RM; ++t)
                            a[q][t] = elem_at<KIND>(s, row[t] + min(reg_col<NW, CPW>(qc + q, 0, wave), n - 1) * n, w, w2);
                } else {
#pragma unroll
                    for (int q = 0; q < QC; ++q)
#pragma unroll
                        for (int t = 0; t < RM; ++t) a[q][t] = czero<double>();
                }
#pragma unroll
                for (int q = 0; q < QC; ++q)
#pragma unroll
                    for (int t = 0; t < RM; ++t) {
                        const bool ok = in[t] && reg_col<NW, CPW>(qc + q, 0, wave) < n;
                        a[q][t].re = ok ? a[q][t].re : 0.0;
                        a[q][t].im = ok ? a[q][t].im : 0.0;
                        if (any) asum[t] += zabs(a[q][t]);
                        x[qc + q][t] = to_t<float>(a[q][t]);
                    }
                __builtin_amdgcn_sched_barrier(0);  // one chunk's operator loads in flight at a time
            }
        });
    }
    double* ap = reinterpret_cast<double*>(parts);
#pragma unroll
    for (int t = 0; t < RM; ++t)
        if (in[t]) ap[wave * n + row[t]] = asum[t];
    if (tid == 0) R.sc[12] = 0;
    int lpos[RM];
    C b[1][RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        lpos[t] = in[t] ? row[t] : -1;
        b[0][t] = czero<float>();
    }
    __syncthreads();
    double an = 0.0;
#pragma unroll
    for (int t = 0; t < RM; ++t) an = nmax(an, (ap[row[t]] + ap[n + row[t]]) + (ap[2 * n + row[t]] + ap[3 * n + row[t]]));
    const double anorm = wave_dmax(an);
    const int rot = reg_eliminate<float, NW, RM, CPW, 0, true, RM == 1, false>(x, b, 0, lpos, n, R);
    C rsc[RM];  // row r of the inverse is rsc times the register row
#pragma unroll
    for (int t = 0; t < RM; ++t) rsc[t] = ldc<3>(R.rp + max(lpos[t], 0));
    const SysDesc s = reg_sys(sp, fidx);
    const double w = s.freq ? kTwoPi * s.freq[fidx] : 0.0, w2 = w * w;
    const int info = R.sc[12];
    if (info != 0) {
        reg_singular(s, fidx, info, NW * 64);
        return;
    }
    // ---- solve and refine, four right-hand sides at a time
    int it_max = 0;
    bool ok = true;
    z64* p64 = reinterpret_cast<z64*>(parts);  // [wave][g][row]
    C* p32 = reinterpret_cast<C*>(parts);
    for (int g0 = 0; g0 < s.nrhs; g0 += G) {
        const int gc = min(G, s.nrhs - g0);
        const bool act = wave < gc;
        const double2* Fg = s.F + (size_t)(g0 + min(wave, gc - 1)) * s.ldf;
        z64 r[RM], xr[RM];
#pragma unroll
        for (int t = 0; t < RM; ++t) {
            const z64 f = ldc<1>(reinterpret_cast<const z64*>(Fg) + row[t]);
            r[t] = cmk<double>(in[t] ? f.re : 0.0, in[t] ? f.im : 0.0);
            xr[t] = czero<double>();
        }
        const double bmax = wave_zmax<RM>(r);
        double be = 0.0;
        int it = -1;
        bool conv = false;
        for (;;) {
            // the residual scaled by a power of two into complex64's range, in the order of
            // the inverse's columns
            double c1 = 0.0;
#pragma unroll
            for (int t = 0; t < RM; ++t) c1 = nmax(c1, cabs1(r[t]));
            c1 = wave_dmax(c1);
            const int ex = (c1 > 0.0 && c1 < __builtin_inf()) ? __builtin_amdgcn_frexp_exp(c1) : 0;
#pragma unroll
            for (int t = 0; t < RM; ++t)
                if (in[t])
                    stc<3>(rv + (lpos[t] * G + wave), cmk<float>((float)__builtin_amdgcn_ldexp(r[t].re, -ex),
                                                                 (float)__builtin_amdgcn_ldexp(r[t].im, -ex)));
            if (lane == 0) ds[wave] = act ? be : 0.0;
            __syncthreads();
            if (it >= 0) {
                conv = true;
#pragma unroll
                for (int g = 0; g < G; ++g)
                    if (!(ds[g] <= kp.tol)) conv = false;
                if (conv || it >= kp.max_iter) break;
            }
            // ---- d = A^-1 r: this wavefront's columns
            C acc[RM][G];
#pragma unroll
            for (int t = 0; t < RM; ++t)
#pragma unroll
                for (int g = 0; g < G; ++g) acc[t][g] = czero<float>();
#pragma unroll
            for (int i = 0; i < CPW; ++i) {
                const int c = reg_col<NW, CPW>(i, rot, wave);
                if (c < n) {
                    C v[G];
#pragma unroll
                    for (int g = 0; g < G; ++g) v[g] = ldc<3>(rv + (c * G + g));
#pragma unroll
                    for (int t = 0; t < RM; ++t)
#pragma unroll
                        for (int g = 0; g < G; ++g) cfma(acc[t][g], x[i][t], v[g]);
                }
            }
#pragma unroll
            for (int t = 0; t < RM; ++t)
                if (in[t])
#pragma unroll
                    for (int g = 0; g < G; ++g) stc<3>(p32 + ((wave * G + g) * n + row[t]), acc[t][g]);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                C d = czero<float>();
#pragma unroll
                for (int v = 0; v < NW; ++v) {
                    const C e = ldc<3>(p32 + ((v * G + wave) * n + row[t]));
                    d.re += e.re;
                    d.im += e.im;
                }
                d = cmul(d, rsc[t]);
                xr[t].re += __builtin_amdgcn_ldexp((double)d.re, ex);
                xr[t].im += __builtin_amdgcn_ldexp((double)d.im, ex);
                if (in[t]) stc<3>(xs + (wave * n + lpos[t]), xr[t]);
                else xr[t] = czero<double>();
            }
            ++it;
            __syncthreads();
            // ---- r = F - A(w) x in FP64, columns split over the wavefronts
            z64 ra[RM][G];
#pragma unroll
            for (int t = 0; t < RM; ++t)
#pragma unroll
                for (int g = 0; g < G; ++g) ra[t][g] = czero<double>();
            with_kind(s, [&](auto kc) {
                constexpr int KIND = decltype(kc)::value;
                constexpr int QC = RM == 1 || KIND == kOpOne ? 4 : 2;
                for (int c0 = QC * wave; c0 < n; c0 += NW * QC) {
                    z64 a[QC][RM];
#pragma unroll
                    for (int q = 0; q < QC; ++q)
#pragma unroll
                        for (int t = 0; t < RM; ++t)
                            a[q][t] = elem_at<KIND>(s, row[t] + min(c0 + q, n - 1) * n, w, w2);
#pragma unroll
                    for (int q = 0; q < QC; ++q) {
                        const int c = c0 + q;
                        if (c < n) {
#pragma unroll
                            for (int g = 0; g < G; ++g)
                                if (g < gc) {
                                    const z64 v = ldc<3>(xs + (g * n + c));
#pragma unroll
                                    for (int t = 0; t < RM; ++t) cfma(ra[t][g], a[q][t], v);
                                }
                        }
                    }
                }
            });
#pragma unroll
            for (int t = 0; t < RM; ++t)
                if (in[t])
#pragma unroll
                    for (int g = 0; g < G; ++g) stc<3>(p64 + ((wave * G + g) * n + row[t]), ra[t][g]);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const z64 f = ldc<1>(reinterpret_cast<const z64*>(Fg) + row[t]);
                z64 a = czero<double>();
#pragma unroll
                for (int v = 0; v < NW; ++v) {
                    const z64 e = ldc<3>(p64 + ((v * G + wave) * n + row[t]));
                    a.re += e.re;
                    a.im += e.im;
                }
                r[t] = cmk<double>(in[t] ? f.re - a.re : 0.0, in[t] ? f.im - a.im : 0.0);
            }
            be = backward_error(wave_zmax<RM>(r), anorm, wave_zmax<RM>(xr), bmax);
        }
        if (!conv) ok = false;
        if (it > it_max) it_max = it;
        if (s.X && act) {
            double2* X = s.X + (size_t)fidx * s.ldx * s.nrhs + (size_t)(g0 + wave) * s.ldx;
#pragma unroll
            for (int t = 0; t < RM; ++t)
                if (in[t]) st_z(X + row[t], ldc<3>(xs + (wave * n + row[t])));
        }
        if (s.berr && act && lane == 0) s.berr[(size_t)fidx * s.nrhs + g0 + wave] = be;
        if (s.C) project_cols<NW * 64>(s, fidx, xs, g0, gc);
        __syncthreads();
    }
    if (tid == 0) {
        s.info[fidx] = ok ? 0 : -1;
        if (s.iters) s.iters[fidx] = it_max;
    }
}

// ==== complex128 LU ================================================================================
// Triangular substitution by one wavefront, v[t] = entry lane + 64 t of the
// vector.  BACK: unknowns n-1 .. 0, else 0 .. n-1.  at(k, i): the coefficient of
// unknown k in equation i (used for i on the far side of k only, clamped otherwise);
// diag(k): the reciprocal of the diagonal.  KEEP: unknowns are kept apart as they are found.  (Without,
// those found have zero times the current unknown subtracted, which is NaN where that one
// overflowed; the adjoint, whose sums are not finite then either way, saves the registers.)
// Blocks of KB unknowns, the next
// block's coefficients loaded ahead of the chain.
template <int RM, bool BACK, bool UNIT, bool KEEP = false, typename FA, typename FD>
__device__ __forceinline__ void wave_substitute(z64 (&v)[RM], int n, FA&& at, FD&& diag) {
    constexpr int KB = RM == 1 ? 4 : 2;
    const int lane = threadIdx.x & 63;
    z64 a[2][KB][RM], d[2][KB], x[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) x[t] = v[t];
    auto load = [&](int k0, z64 (&la)[KB][RM], z64 (&ld)[KB]) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
            const int k = BACK ? max(k0 - u, 0) : min(k0 + u, n - 1);  // beyond the end: read, not used
#pragma unroll
            for (int t = 0; t < RM; ++t) la[u][t] = at(k, lane + 64 * t);
            if (!UNIT) ld[u] = diag(k);
        }
    };
    auto step = [&](int k0, z64 (&la)[KB][RM], z64 (&ld)[KB]) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
            const int k = BACK ? k0 - u : k0 + u;
            if (BACK ? k < 0 : k >= n) break;
            const int lk = k & 63, tk = k >> 6;
            z64 vk = v[0];
#pragma unroll
            for (int t = 1; t < RM; ++t)
                if (tk == t) vk = v[t];
            vk = cbcast(vk, lk);
            if (!UNIT) vk = cmul(vk, ld[u]);
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const int i = lane + 64 * t;
                if (KEEP) {  // entries already found are updated too, and no longer read
                    x[t].re = i == k ? vk.re : x[t].re;
                    x[t].im = i == k ? vk.im : x[t].im;
                    cfms(v[t], la[u][t], vk);
                } else {
                    const bool far = BACK ? i < k : i > k;
                    z64 c = la[u][t];
                    c.re = far ? c.re : 0.0;
                    c.im = far ? c.im : 0.0;
                    if (!UNIT && i == k) v[t] = vk;
                    cfms(v[t], c, vk);
                }
            }
        }
    };
    const int dir = BACK ? -1 : 1;
    int k = BACK ? n - 1 : 0;
    load(k, a[0], d[0]);
    for (int b0 = 0; b0 < n; b0 += 2 * KB, k += 2 * KB * dir) {
        load(k + KB * dir, a[1], d[1]);
        step(k, a[0], d[0]);
        load(k + 2 * KB * dir, a[0], d[0]);
        step(k + KB * dir, a[1], d[1]);
    }
    if (KEEP)
#pragma unroll
        for (int t = 0; t < RM; ++t) v[t] = x[t];
}

// sum over the wavefront, in every lane
__device__ __forceinline__ double wave_dsum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// ---- backward errors of solutions in registers and (vec, [wavefront][n]) in LDS ---------------------
// Right-hand side g by this wavefront alone: r = F - A(w) x and the row sums of |A|.
template <int RM>
__device__ __forceinline__ void reg_berr_wave(const SysDesc& s, int fidx, double w, double w2, int g, const z64 (&v)[RM], const z64* vw) {
    const int n = __builtin_amdgcn_readfirstlane(s.n), lane = threadIdx.x & 63;
    int row[RM];
    bool in[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        in[t] = lane + 64 * t < n;
        row[t] = in[t] ? lane + 64 * t : n - 1;
    }
    const z64* Fg = reinterpret_cast<const z64*>(s.F) + (size_t)g * s.ldf;
    z64 r[RM], f[RM], xv[RM];
    double as[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        f[t] = ldc<1>(Fg + row[t]);
        f[t].re = in[t] ? f[t].re : 0.0;
        f[t].im = in[t] ? f[t].im : 0.0;
        r[t] = f[t];
        xv[t] = cmk<double>(in[t] ? v[t].re : 0.0, in[t] ? v[t].im : 0.0);
        as[t] = 0.0;
    }
    with_kind<false>(s, [&](auto kc) {
        constexpr int KIND = decltype(kc)::value;
        for (int c0 = 0; c0 < n; c0 += 4) {
            z64 a[4][RM];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    a[q][t] = elem_at<KIND>(s, row[t] + min(c0 + q, n - 1) * n, w, w2);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c0 + q < n) {
                    const z64 xc = ldc<3>(vw + c0 + q);
#pragma unroll
                    for (int t = 0; t < RM; ++t) {
                        as[t] += zabs(a[q][t]);
                        cfms(r[t], a[q][t], xc);
                    }
                }
        }
    });
    double an = 0.0;
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        an = nmax(an, as[t]);
        r[t].re = in[t] ? r[t].re : 0.0;
        r[t].im = in[t] ? r[t].im : 0.0;
    }
    const double be = backward_error(wave_zmax<RM>(r), wave_dmax(an), wave_zmax<RM>(xv), wave_zmax<RM>(f));
    if (lane == 0) s.berr[(size_t)fidx * s.nrhs + g] = be;
}

// Right-hand sides g0 .. g0 + na - 1 (na <= NW / 2, the last of the point) by every wavefront:
// columns split over them, partial sums in LDS (part: NW (2 na + 1) n doubles, where U was).
// One wavefront per right-hand side left the others idle for a pass over A(w) with one
// column batch in flight (n = 128 with D, 1 right-hand side, 1024 points: 1047 us, 919 now).
template <int NW, int RM>
__device__ __forceinline__ void reg_berr_joint(const SysDesc& s, int fidx, double w, double w2, int g0, int na, const z64 (&v)[RM],
                                               const z64* vec, z64* part) {
    constexpr int NA = NW / 2;
    const int n = __builtin_amdgcn_readfirstlane(s.n), lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double* asums = reinterpret_cast<double*>(part + (size_t)NW * na * n);  // [wavefront][n]
    int row[RM];
    bool in[RM];
    z64 acc[RM][NA];
    double as[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        in[t] = lane + 64 * t < n;
        row[t] = in[t] ? lane + 64 * t : n - 1;
        as[t] = 0.0;
#pragma unroll
        for (int g = 0; g < NA; ++g) acc[t][g] = czero<double>();
    }
    __syncthreads();  // every solution is in LDS, U is free
    with_kind(s, [&](auto kc) {
        constexpr int KIND = decltype(kc)::value;
        for (int c0 = 4 * wave; c0 < n; c0 += 4 * NW) {
            z64 a[4][RM];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < RM; ++t) a[q][t] = elem_at<KIND>(s, row[t] + min(c0 + q, n - 1) * n, w, w2);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c0 + q < n) {
#pragma unroll
                    for (int t = 0; t < RM; ++t) as[t] += zabs(a[q][t]);
#pragma unroll
                    for (int g = 0; g < NA; ++g)
                        if (g < na) {
                            const z64 x = ldc<3>(vec + (g * n + c0 + q));
#pragma unroll
                            for (int t = 0; t < RM; ++t) cfma(acc[t][g], a[q][t], x);
                        }
                }
        }
    });
#pragma unroll
    for (int t = 0; t < RM; ++t)
        if (in[t]) {
            asums[wave * n + row[t]] = as[t];
#pragma unroll
            for (int g = 0; g < NA; ++g)
                if (g < na) stc<3>(part + ((wave * na + g) * n + row[t]), acc[t][g]);
        }
    __syncthreads();
    if (wave >= na) return;
    const z64* Fg = reinterpret_cast<const z64*>(s.F) + (size_t)(g0 + wave) * s.ldf;
    z64 r[RM], f[RM], xv[RM];
    double an = 0.0;
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        f[t] = ldc<1>(Fg + row[t]);
        z64 a = czero<double>();
        double sa = 0.0;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            const z64 p = ldc<3>(part + ((q * na + wave) * n + row[t]));
            a.re += p.re;
            a.im += p.im;
            sa += asums[q * n + row[t]];
        }
        an = nmax(an, sa);
        r[t] = cmk<double>(in[t] ? f[t].re - a.re : 0.0, in[t] ? f[t].im - a.im : 0.0);
        f[t].re = in[t] ? f[t].re : 0.0;
        f[t].im = in[t] ? f[t].im : 0.0;
        xv[t] = cmk<double>(in[t] ? v[t].re : 0.0, in[t] ? v[t].im : 0.0);
    }
    const double be = backward_error(wave_zmax<RM>(r), wave_dmax(an), wave_zmax<RM>(xv), wave_zmax<RM>(f));
    if (lane == 0) s.berr[(size_t)fidx * s.nrhs + g0 + wave] = be;
}

// BERR: with backward errors.
template <int NW, int RM, int CPW, bool ADJ, bool BERR>
__device__ __forceinline__ void reg_point_plain(const SysDesc* sp, int fidx, const KParams& kp, char* smem) {
    constexpr int NE = 2;  // right-hand sides per wavefront and factorisation
    constexpr int NA = NW / 2;  // up to here the backward errors are every wavefront's work
    const int n = __builtin_amdgcn_readfirstlane(sp->n), tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrhs = __builtin_amdgcn_readfirstlane(sp->nrhs);
    constexpr bool adj = ADJ;
    RegLds<double> R;
    char* p = smem;
    R.sc = reinterpret_cast<int*>(p);
    p += 64;
    R.rp = reinterpret_cast<z64*>(p);
    p += 16 * n;
    R.pos = reinterpret_cast<int*>(p);
    p += align16(n * 4LL);
    // multiplier columns; after the elimination one vector per wavefront
    R.lcol = reinterpret_cast<z64*>(p);
    z64* vec = R.lcol;  // [wave][n]
    p += 16 * (NW == 8 ? 12 : 8) * n;
    z64* nu = reinterpret_cast<z64*>(p);  // adjoint: nu, then xi
    p += adj ? 32 * n : 0;
    R.U = reinterpret_cast<z64*>(p);
    p += reg_packed_bytes(n, NW, adj);
    double* red = reinterpret_cast<double*>(p);  // adjoint: 2 NW doubles
    int row[RM];
    bool in[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        in[t] = lane + 64 * t < n;
        row[t] = in[t] ? lane + 64 * t : n - 1;
    }
    double accJ = 0.0;
    z64 xi[RM];  // adjoint: this wavefront's part of sum_r conj(g_r) x_r
#pragma unroll
    for (int t = 0; t < RM; ++t) xi[t] = czero<double>();
    // more right-hand sides than the extra columns hold: the factorisation is repeated
    for (int g0 = 0; g0 < nrhs; g0 += NW * NE) {
        const int gn = min(NW * NE, nrhs - g0), ne = (gn + NW - 1) / NW;
        const bool last = g0 + NW * NE >= nrhs;
        z64 x[CPW][RM], b[NE][RM];
        int lpos[RM];
        {
            const SysDesc s = reg_sys(sp, fidx);
            const double w = s.freq ? kTwoPi * s.freq[fidx] : 0.0, w2 = w * w;
            with_kind<false>(s, [&](auto kc) {
                constexpr int KIND = decltype(kc)::value;
#pragma unroll
                for (int qc = 0; qc < CPW; qc += 4) {
                    if (reg_col<NW, CPW>(qc, 0, wave) < n) {
#pragma unroll
                        for (int q = qc; q < qc + 4; ++q)
#pragma unroll
                            for (int t = 0; t < RM; ++t)
                                x[q][t] = elem_at<KIND>(s, row[t] + min(reg_col<NW, CPW>(q, 0, wave), n - 1) * n, w, w2);
                    } else {
#pragma unroll
                        for (int q = qc; q < qc + 4; ++q)
#pragma unroll
                            for (int t = 0; t < RM; ++t) x[q][t] = czero<double>();
                    }
                    __builtin_amdgcn_sched_barrier(0);  // one chunk's operator loads in flight at a time
                }
            });
#pragma unroll
            for (int q = 0; q < CPW; ++q)
#pragma unroll
                for (int t = 0; t < RM; ++t) {
                    const bool ok = in[t] && reg_col<NW, CPW>(q, 0, wave) < n;
                    x[q][t].re = ok ? x[q][t].re : 0.0;
                    x[q][t].im = ok ? x[q][t].im : 0.0;
                }
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int t = 0; t < RM; ++t) {
                    b[e][t] = czero<double>();
                    if (e < ne) {
                        const int g = g0 + min(e * NW + wave, gn - 1);
                        const z64 f = ldc<1>(reinterpret_cast<const z64*>(s.F) + (row[t] + (size_t)g * s.ldf));
                        b[e][t] = cmk<double>(in[t] ? f.re : 0.0, in[t] ? f.im : 0.0);
                    }
                }
        }
#pragma unroll
        for (int t = 0; t < RM; ++t) lpos[t] = in[t] ? row[t] : -1;
        if (tid == 0) R.sc[12] = 0;
        __syncthreads();
        const int rot = reg_eliminate<double, NW, RM, CPW, NE, false, NW == 8, ADJ>(x, b, ne, lpos, n, R);
        const SysDesc s = reg_sys(sp, fidx);
        const double w = s.freq ? kTwoPi * s.freq[fidx] : 0.0, w2 = w * w;
        const bool want_berr = BERR && s.berr != nullptr;
        const int info = R.sc[12];
        if (info != 0) {
            reg_singular(s, fidx, info, NW * 64);
            return;
        }
        // ---- back substitution: wavefront w, right-hand sides w, w + NW, ...
        auto u_at = [&](int k, int i) { return ldc<3>(R.U + (((k * (k + 1)) >> 1) + min(i, k))); };
        auto u_rd = [&](int k) { return ldc<3>(R.rp + k); };
        z64* vw = vec + (size_t)wave * n;
        for (int e = 0; e < ne; ++e) {
            const int g = g0 + e * NW + wave;
            const bool act = e * NW + wave < gn;
            z64 v[RM];
            if (act) {
#pragma unroll
                for (int t = 0; t < RM; ++t) {
                    z64 y = b[0][t];
#pragma unroll
                    for (int q = 1; q < NE; ++q)
                        if (e == q) y = b[q][t];
                    if (in[t]) stc<3>(vw + lpos[t], y);
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int t = 0; t < RM; ++t) v[t] = ldc<3>(vw + row[t]);
                wave_substitute<RM, true, false, !ADJ>(v, n, u_at, u_rd);
                if (s.X) {
                    double2* X = s.X + (size_t)fidx * s.ldx * s.nrhs + (size_t)g * s.ldx;
#pragma unroll
                    for (int t = 0; t < RM; ++t)
                        if (in[t]) st_z(X + row[t], v[t]);
                }
                if (want_berr || s.C) {
#pragma unroll
                    for (int t = 0; t < RM; ++t)
                        if (in[t]) stc<3>(vw + row[t], v[t]);
                    __builtin_amdgcn_wave_barrier();
                }
                if constexpr (adj) {  // g_r = c^H x_r, J += |g_r|^2, xi += conj(g_r) x_r
                    double re = 0.0, im = 0.0;
#pragma unroll
                    for (int t = 0; t < RM; ++t)
                        if (in[t]) {
                            const z64 c = ldc<1>(reinterpret_cast<const z64*>(s.c) + row[t]);
                            re += c.re * v[t].re + c.im * v[t].im;
                            im += c.re * v[t].im - c.im * v[t].re;
                        }
                    const z64 gr = cmk<double>(wave_dsum(re), wave_dsum(im));
                    accJ += gr.re * gr.re + gr.im * gr.im;
#pragma unroll
                    for (int t = 0; t < RM; ++t)
                        if (in[t]) cfma(xi[t], cconj(gr), v[t]);
                }
            }
            if (want_berr) {
                const int na = min(NW, gn - e * NW);
                if (na <= NA && n + 1 >= NW * (2 * na + 1)) reg_berr_joint<NW, RM>(s, fidx, w, w2, g0 + e * NW, na, v, vec, R.U);
                else if (act) reg_berr_wave<RM>(s, fidx, w, w2, g, v, vw);
            }
            if (s.C) {
                __syncthreads();
                project_cols<NW * 64>(s, fidx, vec, g0 + e * NW, min(NW, gn - e * NW));
                __syncthreads();
            }
        }
        if (adj && last) {
            // ---- nu = A^-H c: U^H z = c, then L^H P nu = z.  mu_r = g_r nu, so
            // sum_r mu_r^H (.) x_r = nu^H (.) xi with xi = sum_r conj(g_r) x_r
            z64* xv = nu + n;
            z64 z[RM];
            if (wave == NW - 1) {
#pragma unroll
                for (int t = 0; t < RM; ++t) z[t] = ldc<1>(reinterpret_cast<const z64*>(s.c) + row[t]);
                wave_substitute<RM, false, false>(
                    z, n, [&](int k, int i) { const int j = min(max(i, k), n - 1); return cconj(ldc<3>(R.U + (((j * (j + 1)) >> 1) + k))); },
                    [&](int k) { return cconj(u_rd(k)); });
            }
#pragma unroll
            for (int t = 0; t < RM; ++t)
                if (in[t]) stc<3>(vw + row[t], xi[t]);
            if (lane == 0) red[wave] = accJ;
            __syncthreads();  // U is free, every wavefront's xi stored
            z64* Lp = R.U;    // L packed by rows: L[i][k] at i (i - 1) / 2 + k
#pragma unroll
            for (int i = 0; i < CPW; ++i) {
                const int c = reg_col<NW, CPW>(i, rot, wave);
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (lpos[t] > c)
                        stc<3>(Lp + (((lpos[t] * (lpos[t] - 1)) >> 1) + c), cmk<double>(-x[i][t].re, -x[i][t].im));
            }
            int* kpos = R.pos;
            if (wave == 0)
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (in[t]) kpos[lpos[t]] = row[t];
            for (int i = tid; i < n; i += NW * 64) {
                z64 a = czero<double>();
                for (int v = 0; v < NW; ++v) {
                    const z64 e = ldc<3>(vec + ((size_t)v * n + i));
                    a.re += e.re;
                    a.im += e.im;
                }
                stc<3>(xv + i, a);
            }
            __syncthreads();
            if (wave == NW - 1) {
                wave_substitute<RM, true, true>(
                    z, n, [&](int k, int i) { return cconj(ldc<3>(Lp + (k > 0 ? ((k * (k - 1)) >> 1) + min(i, k - 1) : 0))); },
                    [&](int) { return czero<double>(); });
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (in[t]) stc<3>(nu + kpos[row[t]], z[t]);
            }
            __syncthreads();
            // ---- nu^H K xi: rows over the lanes, columns over the wavefronts
            double ei = 0.0;
            {
                z64 kx[RM];
#pragma unroll
                for (int t = 0; t < RM; ++t) kx[t] = czero<double>();
                for (int c0 = wave; c0 < n; c0 += 4 * NW) {
                    z64 k[4][RM];
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int t = 0; t < RM; ++t) {
                            const int e = row[t] + min(c0 + NW * q, n - 1) * n;
                            k[q][t] = s.real_ops ? cmk<double>(lds1<1>(s.K + e), 0.0) : ldc<1>(reinterpret_cast<const z64*>(s.K) + e);
                        }
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (c0 + NW * q < n) {
                            const z64 v = ldc<3>(xv + c0 + NW * q);
#pragma unroll
                            for (int t = 0; t < RM; ++t) cfma(kx[t], k[q][t], v);
                        }
                }
#pragma unroll
                for (int t = 0; t < RM; ++t)
                    if (in[t]) {
                        ei += cmul(cconj(ldc<3>(nu + row[t])), kx[t]).im;
                    }
            }
            ei = wave_dsum(ei);
            if (lane == 0) red[NW + wave] = ei;
            // ---- the modal products phi_k^T nu and phi_k^T xi: k over the lanes (64 at a
            // time, Phi^T read along k), rows over the wavefronts
            double* out = s.adj_out + (size_t)fidx * (s.p + 2);
            double* mp = reinterpret_cast<double*>(Lp);  // [wave][4][64]
            const z64 keta = cmk<double>(1.0, s.eta);
            const int per = (n + NW - 1) / NW, i0 = wave * per, i1 = min(n, i0 + per);
            for (int k0 = 0; k0 < s.p; k0 += 64) {
                const int k = min(k0 + lane, s.p - 1);
                z64 pn = czero<double>(), px = czero<double>();
                for (int ib = i0; ib < i1; ib += 8) {
                    double f[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) f[u] = lds1<1>(s.PhiT + ((size_t)min(ib + u, i1 - 1) * s.p + k));
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (ib + u < i1) {
                            const z64 a = ldc<3>(nu + ib + u), c = ldc<3>(xv + ib + u);
                            pn.re = fma(f[u], a.re, pn.re);
                            pn.im = fma(f[u], a.im, pn.im);
                            px.re = fma(f[u], c.re, px.re);
                            px.im = fma(f[u], c.im, px.im);
                        }
                }
                __syncthreads();  // L (first chunk) and the previous chunk's sums are consumed
                mp[(wave * 4 + 0) * 64 + lane] = pn.re;
                mp[(wave * 4 + 1) * 64 + lane] = pn.im;
                mp[(wave * 4 + 2) * 64 + lane] = px.re;
                mp[(wave * 4 + 3) * 64 + lane] = px.im;
                __syncthreads();
                if (wave == 0 && k0 + lane < s.p) {
                    double a[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        a[q] = mp[q * 64 + lane];
                        for (int v = 1; v < NW; ++v) a[q] += mp[(v * 4 + q) * 64 + lane];
                    }
                    const z64 m = cmul(cmul(keta, cmk<double>(a[0], -a[1])), cmk<double>(a[2], a[3]));
                    out[2 + k] = -2.0 * s.kdiag[k] * m.re;
                }
            }
            __syncthreads();
            if (tid == 0) {
                double J = red[0], E = red[NW];
                for (int v = 1; v < NW; ++v) {
                    J += red[v];
                    E += red[NW + v];
                }
                out[0] = J;
                out[1] = 2.0 * E;  // -2 Re(i nu^H K xi)
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        sp->info[fidx] = 0;
        if (sp->iters) sp->iters[fidx] = 0;
    }
}

// ---- the kernel ------------------------------------------------------------------------------
// MAXR: rows per lane of the launch's largest system (1: n <= 64, 2: n <= 128).
// ADJ: the adjoint (complex128), an instance of its own: it keeps L in registers
// through the substitutions.  BERR: plain with backward errors, an instance of its own too: their
// code costs the solves without them 1 to 4 %, the adjoint 7 to 12 %.
//
// Measured against the kernels it replaced there (us a call): n = 24, 32 points,
// plain 80 -> 39 alone; n = 60, 1000 points, host arrays, plain 557 -> 195 (76 of it by
// the results' way back); n = 64, 4096 explicit matrices 1708 -> 471; n = 47, 1501
// points, 2 right-hand sides, refined 437 -> 103; n = 96 complex operators, 1500
// points, plain 831 -> 677; n = 123, 2048 points, 4 right-hand sides, refined
// 1698 -> 1381; the adjoint at n = 128, 2048 points 2627 -> 1900.
template <typename T, int MAXR, bool ADJ, bool BERR>
__global__ void __launch_bounds__(64 * reg_waves(sizeof(T) == 4, MAXR))
    __attribute__((amdgpu_waves_per_eu(MAXR == 1 ? 4 : 2, MAXR == 1 ? 4 : 2)))
reg_kernel(KParams kp) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int s_item;
    const int tid = threadIdx.x;
    // one system: points dealt round-robin (equal work; no queue to reset);
    // a batch takes points from the queue
    int item = blockIdx.x;
    for (;;) {
        if (kp.items) {
            if (tid == 0) s_item = atomicAdd(kp.counter, 1);
            __syncthreads();
            item = s_item;
        }
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= kp.nitems) break;
        int sysi = 0, fidx = item;
        if (kp.items) {
            const int2 it = kp.items[item];
            sysi = __builtin_amdgcn_readfirstlane(it.x);
            fidx = __builtin_amdgcn_readfirstlane(it.y);
        }
        // a single system's descriptor is read from the kernel arguments where they lie
        const SysDesc* sp = kp.sys ? kp.sys + sysi
                                   : &((const KParams*)__builtin_amdgcn_kernarg_segment_ptr())->one;
        const int n = __builtin_amdgcn_readfirstlane(sp->n);
        if constexpr (sizeof(T) == 4) {
            if constexpr (MAXR == 1) {
                if (n <= 32) reg_point_refined<1, 8>(sp, fidx, kp, smem);
                else reg_point_refined<1, 16>(sp, fidx, kp, smem);
            } else {
                if (n <= 64) reg_point_refined<1, 16>(sp, fidx, kp, smem);
                else if (n <= 96) reg_point_refined<2, 24>(sp, fidx, kp, smem);
                else reg_point_refined<2, 32>(sp, fidx, kp, smem);
            }
        } else {
            if constexpr (MAXR == 1) {
                if (n <= 32) reg_point_plain<4, 1, 8, ADJ, BERR>(sp, fidx, kp, smem);
                else reg_point_plain<4, 1, 16, ADJ, BERR>(sp, fidx, kp, smem);
            } else {
                if (!ADJ && n <= 64) reg_point_plain<8, 1, 8, false, BERR>(sp, fidx, kp, smem);  // in a batch
                else if (n <= 96) reg_point_plain<8, 2, 12, ADJ, BERR>(sp, fidx, kp, smem);
                else reg_point_plain<8, 2, 16, ADJ, BERR>(sp, fidx, kp, smem);
            }
        }
        __syncthreads();
        item += gridDim.x;
    }
}

}  // namespace stc
