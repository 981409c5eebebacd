// stc_wide.h -- wide-panel blocked LU of the sweep kernel (gfx950).
//
// The blocked path of sweep_kernel<T, MAXR, 1> (<T, MAXR, 2>: Gauss 3M products in the
// panels' update).  It factors A(w) in the workgroup's global factor slot, left-looking,
// in steps of 32 columns (complex64) or 16 (complex128), with panels of jb columns (a
// step, or half a complex64 one) held in LDS, one or two workgroups per CU:
//
//   step: its columns, assembled from the operators, are brought up to date with all
//   finished columns in the MFMA accumulators of the workgroup (left_update) and
//   go to the LDS panel (m rows x jb columns, logical row order):
//     per 16-column sub-panel: pivoted LU with the rows distributed over the
//     threads (a thread's rows in registers, one barrier per
//     column), rows permuted in the LDS panel afterwards; the 16 x 16
//     unit-lower diagonal block inverted (one entry per thread); the panel's
//     remaining columns updated on MFMA (U rows = Linv A, rows below -= L21 U);
//   the first right-hand sides are the last step's columns, without a panel.
//
// Rows never move in the slot (row map, as in the 16-column path); only the
// LDS panel is kept in logical order.  Complex products take four real MFMAs
// (three in the Gauss form).
//
// MFMA operand layout used throughout (16x16x4, one wavefront; li = lane % 16,
// lg = lane / 16): lane supplies A[li][k-slot lg] and B[k-slot lg][li]; the
// accumulator register r holds D[row(lg, r)][li].  The k index of step s of a
// 16-block is kk(lg, s) = row(lg, s), so a block's accumulator is directly the
// B (or A) operand of the next product: no register shuffles.
#pragma once

namespace stc {

// d += a * b (complex; a from the lane's A operand, b its B operand).
template <typename T>
__device__ __forceinline__ void cmfma(typename Mfma<T>::acc& dre, typename Mfma<T>::acc& dim, cx<T> a,
                                      T bre, T bim) {
    using M = Mfma<T>;
    dre = M::run(a.re, bre, dre);
    dre = M::run(-a.im, bim, dre);
    dim = M::run(a.re, bim, dim);
    dim = M::run(a.im, bre, dim);
}

// Gauss (3M) form of d += a * b over three accumulators: x += a_r b_r,
// y += a_i b_i, z += (a_r + a_i)(b_r + b_i); with x, y, z started at (d_r, 0,
// d_r + d_i) the result is d_r = x - y, d_i = z - x - y.  Three real products
// instead of four.
template <typename T>
__device__ __forceinline__ void cmfma3(typename Mfma<T>::acc& x, typename Mfma<T>::acc& y,
                                       typename Mfma<T>::acc& z, cx<T> a, T asum, T bre, T bim) {
    using M = Mfma<T>;
    x = M::run(a.re, bre, x);
    y = M::run(a.im, bim, y);
    z = M::run(asum, bre + bim, z);
}

template <typename T>
__device__ __forceinline__ void acc_zero(typename Mfma<T>::acc& a) {
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = T(0);
}


// ---- branch-free pivot search of one wavefront -----------------------------------------------
// A candidate row is the pair (hk, lo), compared lexicographically: hk orders
// |re| + |im| with LAPACK izamax's NaN rule (as pivot_key: a NaN in the first
// eligible row wins, a NaN elsewhere is never chosen; 0 = not a candidate),
// lo = (1023 - logical position) << 10 | gather position, so ties go to the
// first row in LAPACK order and the winner's location rides along.
__device__ __forceinline__ unsigned long long pivot_ukey(float v, bool first) {
    return v == v ? (unsigned long long)__float_as_uint(v) + 2ull : (first ? 0x7F800002ull : 1ull);
}
__device__ __forceinline__ unsigned long long pivot_ukey(double v, bool first) {
    return v == v ? (unsigned long long)__double_as_longlong(v) + 2ull : (first ? 0x7FF0000000000002ull : 1ull);
}
template <int CTRL, int RM>
__device__ __forceinline__ unsigned dppu(unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, RM, 0xF, false);
}
template <int CTRL, int RM>
__device__ __forceinline__ void argmax_step(unsigned long long& hk, unsigned& lo) {
    const unsigned long long ok = ((unsigned long long)dppu<CTRL, RM>((unsigned)(hk >> 32)) << 32) |
                                  dppu<CTRL, RM>((unsigned)hk);
    const unsigned ol = dppu<CTRL, RM>(lo);
    const bool better = ok > hk || (ok == hk && ol > lo);
    hk = better ? ok : hk;
    lo = better ? ol : lo;
}
constexpr int kDppRowBcast15 = 0x142;  // lane 15 of each row -> the next row
constexpr int kDppRowBcast31 = 0x143;  // lane 31 -> rows 2 and 3
// Maximum over the wave, returned in every lane: four DPP steps give each
// row of 16 lanes its maximum, two row broadcasts carry it to lane 63.
__device__ __forceinline__ void wave_argmax_packed(unsigned long long& hk, unsigned& lo) {
    argmax_step<kDppXor1, 0xF>(hk, lo);
    argmax_step<kDppXor2, 0xF>(hk, lo);
    argmax_step<kDppHalfMirror, 0xF>(hk, lo);
    argmax_step<kDppMirror, 0xF>(hk, lo);
    argmax_step<kDppRowBcast15, 0xA>(hk, lo);
    argmax_step<kDppRowBcast31, 0xC>(hk, lo);
    const unsigned h = (unsigned)__builtin_amdgcn_readlane((int)(hk >> 32), 63);
    const unsigned l = (unsigned)__builtin_amdgcn_readlane((int)hk, 63);
    hk = ((unsigned long long)h << 32) | l;
    lo = (unsigned)__builtin_amdgcn_readlane((int)lo, 63);
}
// complex64 keys fit one 64-bit word: the 32-bit magnitude key above the
// 20-bit position word (lo < 2^20), so the lexicographic order is the integer
// order and a DPP step moves two dwords instead of three.
template <int CTRL, int RM>
__device__ __forceinline__ void argmax_step64(unsigned long long& v) {
    const unsigned long long o = ((unsigned long long)dppu<CTRL, RM>((unsigned)(v >> 32)) << 32) |
                                 dppu<CTRL, RM>((unsigned)v);
    v = o > v ? o : v;
}
__device__ __forceinline__ void wave_argmax64(unsigned long long& v) {
    argmax_step64<kDppXor1, 0xF>(v);
    argmax_step64<kDppXor2, 0xF>(v);
    argmax_step64<kDppHalfMirror, 0xF>(v);
    argmax_step64<kDppMirror, 0xF>(v);
    argmax_step64<kDppRowBcast15, 0xA>(v);
    argmax_step64<kDppRowBcast31, 0xC>(v);
    const unsigned h = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), 63);
    const unsigned l = (unsigned)__builtin_amdgcn_readlane((int)v, 63);
    v = ((unsigned long long)h << 32) | l;
}
// maximum over the wavefront of one word, uniform
template <int CTRL, int RM>
__device__ __forceinline__ unsigned umax_step(unsigned v) {
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xF, false);
    return o > v ? o : v;
}
__device__ __forceinline__ unsigned wave_umax(unsigned v) {
    v = umax_step<kDppXor1, 0xF>(v);
    v = umax_step<kDppXor2, 0xF>(v);
    v = umax_step<kDppHalfMirror, 0xF>(v);
    v = umax_step<kDppMirror, 0xF>(v);
    v = umax_step<kDppRowBcast15, 0xA>(v);
    v = umax_step<kDppRowBcast31, 0xC>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ void stc1i(int* p, int v) { *(__attribute__((address_space(3))) int*)(p) = v; }
__device__ __forceinline__ void stc1u(unsigned* p, unsigned v) { *(__attribute__((address_space(3))) unsigned*)(p) = v; }

// This wavefront's candidate, uniform: (hk, lo) of the largest, packed in one word for
// complex64 (hk < 2^32).  complex128: one 32-bit maximum of the keys' high words and a
// ballot, the full lexicographic reduction (three words a step) only where rows
// tie there (n = 256 plain 10.9 -> 10.3 ms); complex64 measured 2 % slower so.
template <typename T>
__device__ __forceinline__ unsigned long long wave_candidate(unsigned long long& hk, unsigned& lo) {
    if constexpr (sizeof(T) == 4) {
        unsigned long long pk = (hk << 20) | lo;
        wave_argmax64(pk);
        hk = pk >> 20;
        lo = (unsigned)(pk & 0xFFFFFull);
        return pk;
    } else {
        const unsigned h = hk ? (unsigned)(hk >> 32) + 1u : 0u;
        const unsigned long long b = __ballot(h == wave_umax(h));
        if ((b & (b - 1)) == 0) {
            const int src = __builtin_ctzll(b);
            const unsigned kh = (unsigned)__builtin_amdgcn_readlane((int)(hk >> 32), src);
            const unsigned kl = (unsigned)__builtin_amdgcn_readlane((int)hk, src);
            hk = ((unsigned long long)kh << 32) | kl;
            lo = (unsigned)__builtin_amdgcn_readlane((int)lo, src);
        } else {
            wave_argmax_packed(hk, lo);
        }
        return 0;
    }
}

// Rows moved by a sub-panel's pivoting (the list mvl, sc[12] entries): their
// entries in the other panel columns and in the row map follow; every source
// is read before any destination is written.
template <typename T>
__device__ __forceinline__ void subpanel_moves(cx<T>* __restrict__ P, int ldp, int jbl, int c0, int sbw, int j0,
                                               int* rmap, int* sc, int2* mvl) {
    const int tid = threadIdx.x;
    __syncthreads();
    // permute the moved rows of the other panel columns and of the row map:
    // read every source, then write every destination
    const int cnt = uniform(lds1<3>(sc + 12));
    const int nother = jbl - sbw;  // panel columns outside the sub-panel
    const int per = nother + 1;    // + the row-map entry
    const int total = cnt * per;
    // cnt <= 2 sbw <= 32, and beside a sub-panel lies at most the rest of the widest panel
    constexpr int kMv = (2 * kSB * (wide_jb_max((int)sizeof(cx<T>)) - kSB + 1) + kThreads - 1) / kThreads;
    cx<T> tv[kMv];
    int ti[kMv];
#pragma unroll
    for (int u = 0; u < kMv; ++u) {
        const int e = tid + kThreads * u;
        if (e < total) {
            const int i = e / per, k = e - i * per;
            const int2 mvp = mvl[i];
            if (k == nother) {
                ti[u] = rmap[j0 + mvp.x];
            } else {
                const int c = k < c0 ? k : k + sbw;
                tv[u] = ldc<3>(P + (mvp.x + (size_t)c * ldp));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMv; ++u) {
        const int e = tid + kThreads * u;
        if (e < total) {
            const int i = e / per, k = e - i * per;
            const int2 mvp = mvl[i];
            if (k == nother) {
                rmap[j0 + mvp.y] = ti[u];
            } else {
                const int c = k < c0 ? k : k + sbw;
                stc<3>(P + (mvp.y + (size_t)c * ldp), tv[u]);
            }
        }
    }
    __syncthreads();
}

// ---- 16-column sub-panel of the LDS panel ------------------------------------------------
// Columns [c0, c0 + sbw) of P (m x jb, ld m, logical row order), rows
// [c0, m).  Every thread holds whole rows of the sub-panel (rows
// tid + kThreads t) in registers, x[c] = column c.
// Per column one barrier: each wave finds its best candidate row (packed
// keys, DPP), the winning lane publishes that row's 16 values and the wave's
// key in one of two alternating LDS buffers; after the barrier every thread
// picks the best of the wavefronts' candidates (the same in all), takes the pivot
// row from LDS, scales its own rows' multipliers and applies the rank-1
// update.  Rows stay in their registers; pivots only change their logical
// positions lpos.  Afterwards the sub-panel is stored at its new rows and the
// moved rows of the other panel columns and of rmap[j0 + .] are permuted to
// match (moves listed in mvl).  LAPACK zgetf2 semantics: pivot = first row of
// largest |re| + |im| (izamax, NaN rule of pivot_key), zero pivot: no scaling,
// info = first zero column.  ipiv[j0 + c0 + jj] = 0-based pivot row;
// sc[1] = first zero pivot (1-based).
template <typename T, int MAXR>
__device__ __forceinline__ void subpanel_factor(cx<T>* __restrict__ P, int m, int ldp, int jbl, int c0, int sbw, int j0,
                                                int* ipiv, int* rmap, int* sc, cx<T>* rowbuf, int2* mvl) {
    constexpr int RM = (64 * MAXR + kThreads - 1) / kThreads;  // rows per thread
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mq = m - c0;
    cx<T>* Q = P + c0 + (size_t)c0 * ldp;  // sub-panel origin, ld ldp
    // candidate keys after the row buffers: 2 buffers x kWaves x {key lo, key hi, lo, -}
    unsigned* cand = reinterpret_cast<unsigned*>(rowbuf + 2 * kWaves * kSB);
    cx<T> x[kSB][RM];
    int lpos[RM];
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        const int r = tid + kThreads * t;
        lpos[t] = r < mq ? r : 0x7fffffff;
#pragma unroll
        for (int c = 0; c < kSB; ++c)
            x[c][t] = ldz<3>(Q + (min(r, mq - 1) + (size_t)min(c, sbw - 1) * ldp), c < sbw && r < mq);
    }
    if (tid == 0) stc1i(sc + 12, 0);
    // at most two rows a thread: the column loop unrolled (static register
    // indices, no rotation; n = 256: +3.3 %); four rows: a loop that rotates x
    // so that x[0] is the current column (unrolled, it spills)
    if constexpr (RM <= 2) {
        auto column = [&](auto jc) {
            constexpr int jj = decltype(jc)::value;
            if (jj >= sbw) return;
            const int pb = jj & 1;
            cx<T>* rb = rowbuf + pb * kWaves * kSB;
            unsigned* cb = cand + pb * kWaves * 4;
            unsigned long long hk = 0;
            unsigned lo = 0;
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const bool elig = lpos[t] >= jj && lpos[t] != 0x7fffffff;
                const unsigned long long k = elig ? pivot_ukey(cabs1(x[jj][t]), lpos[t] == jj) : 0ull;
                const unsigned l = elig ? ((unsigned)(1023 - lpos[t]) << 10) | (unsigned)(tid + kThreads * t) : 0u;
                const bool better = k > hk || (k == hk && l > lo);
                hk = better ? k : hk;
                lo = better ? l : lo;
            }
            const unsigned long long pk = wave_candidate<T>(hk, lo);
            const int wg = (int)(lo & 1023u);
            if (hk != 0ull && tid == (wg & (kThreads - 1))) {
                const int tw = wg / kThreads;
#pragma unroll
                for (int c = jj; c < kSB; ++c) {
                    cx<T> v = x[c][0];
#pragma unroll
                    for (int t = 1; t < RM; ++t)
                        if (tw == t) v = x[c][t];
                    stc<3>(rb + (wave * kSB + c), v);
                }
            }
            if (lane == 0) {
                if (sizeof(T) == 4) {
                    *(__attribute__((address_space(3))) unsigned long long*)(cb + wave * 4) = pk;
                } else {
                    stc1u(cb + wave * 4, (unsigned)hk);
                    stc1u(cb + wave * 4 + 1, (unsigned)(hk >> 32));
                    stc1u(cb + wave * 4 + 2, lo);
                }
            }
            __syncthreads();
            unsigned long long bk = 0;
            unsigned bl = 0;
            int bw = 0;
            if (sizeof(T) == 4) {
                unsigned long long bp = 0;
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {
                    const unsigned long long p = *(const __attribute__((address_space(3))) unsigned long long*)(cb + v * 4);
                    const bool better = p > bp;
                    bp = better ? p : bp;
                    bw = better ? v : bw;
                }
                bl = (unsigned)(bp & 0xFFFFFull);
            } else {
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {
                    const unsigned long long k = ((unsigned long long)lds1<3>(cb + v * 4 + 1) << 32) | lds1<3>(cb + v * 4);
                    const unsigned l = lds1<3>(cb + v * 4 + 2);
                    const bool better = k > bk || (k == bk && l > bl);
                    bk = better ? k : bk;
                    bl = better ? l : bl;
                    bw = better ? v : bw;
                }
            }
            bw = __builtin_amdgcn_readfirstlane(bw);
            const int bpos = 1023 - (int)(__builtin_amdgcn_readfirstlane(bl) >> 10);
            const cx<T>* u = rb + bw * kSB;
            const cx<T> pv = ldc<3>(u + jj);
            const bool zero = pv.re == T(0) && pv.im == T(0);
            const cx<T> rp = zero ? czero<T>() : crecip(pv);
            if (tid == 0) {
                stc1i(ipiv + j0 + c0 + jj, j0 + c0 + bpos);
                if (zero && lds1<3>(sc + 1) == 0) stc1i(sc + 1, j0 + c0 + jj + 1);
            }
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                if (lpos[t] == jj) lpos[t] = bpos;
                else if (lpos[t] == bpos) lpos[t] = jj;
            }
            cx<T> uv[kSB];
#pragma unroll
            for (int c = jj + 1; c < kSB; ++c) uv[c] = ldc<3>(u + c);
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                if (lpos[t] > jj && lpos[t] != 0x7fffffff) {
                    const cx<T> l = zero ? x[jj][t] : cmul(x[jj][t], rp);
                    x[jj][t] = l;
#pragma unroll
                    for (int c = jj + 1; c < kSB; ++c) cfms(x[c][t], l, uv[c]);
                }
            }
        };
        static_for(column, std::make_integer_sequence<int, kSB>{});
    } else {
        for (int jj = 0; jj < sbw; ++jj) {
            const int pb = jj & 1;
            cx<T>* rb = rowbuf + pb * kWaves * kSB;
            unsigned* cb = cand + pb * kWaves * 4;
            // ---- this wave's candidate
            unsigned long long hk = 0;
            unsigned lo = 0;
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const bool elig = lpos[t] >= jj && lpos[t] != 0x7fffffff;
                const unsigned long long k = elig ? pivot_ukey(cabs1(x[0][t]), lpos[t] == jj) : 0ull;
                const unsigned l = elig ? ((unsigned)(1023 - lpos[t]) << 10) | (unsigned)(tid + kThreads * t) : 0u;
                const bool better = k > hk || (k == hk && l > lo);
                hk = better ? k : hk;
                lo = better ? l : lo;
            }
            const unsigned long long pk = wave_candidate<T>(hk, lo);
            const int wg = (int)(lo & 1023u);
            if (hk != 0ull && tid == (wg & (kThreads - 1))) {
                const int tw = wg / kThreads;
#pragma unroll
                for (int c = 0; c < kSB; ++c) {
                    cx<T> v = x[c][0];
#pragma unroll
                    for (int t = 1; t < RM; ++t)
                        if (tw == t) v = x[c][t];
                    stc<3>(rb + (wave * kSB + c), v);
                }
            }
            if (lane == 0) {
                if (sizeof(T) == 4) {
                    *(__attribute__((address_space(3))) unsigned long long*)(cb + wave * 4) = pk;
                } else {
                    stc1u(cb + wave * 4, (unsigned)hk);
                    stc1u(cb + wave * 4 + 1, (unsigned)(hk >> 32));
                    stc1u(cb + wave * 4 + 2, lo);
                }
            }
            __syncthreads();
            // ---- the pivot: best of the wavefronts' candidates
            unsigned long long bk = 0;
            unsigned bl = 0;
            int bw = 0;
            if (sizeof(T) == 4) {
                unsigned long long bp = 0;
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {
                    const unsigned long long p = *(const __attribute__((address_space(3))) unsigned long long*)(cb + v * 4);
                    const bool better = p > bp;
                    bp = better ? p : bp;
                    bw = better ? v : bw;
                }
                bl = (unsigned)(bp & 0xFFFFFull);
            } else {
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {
                    const unsigned long long k = ((unsigned long long)lds1<3>(cb + v * 4 + 1) << 32) | lds1<3>(cb + v * 4);
                    const unsigned l = lds1<3>(cb + v * 4 + 2);
                    const bool better = k > bk || (k == bk && l > bl);
                    bk = better ? k : bk;
                    bl = better ? l : bl;
                    bw = better ? v : bw;
                }
            }
            bw = __builtin_amdgcn_readfirstlane(bw);
            const int bpos = 1023 - (int)(__builtin_amdgcn_readfirstlane(bl) >> 10);
            const cx<T>* u = rb + bw * kSB;
            const cx<T> pv = ldc<3>(u);
            const bool zero = pv.re == T(0) && pv.im == T(0);
            const cx<T> rp = zero ? czero<T>() : crecip(pv);
            if (tid == 0) {
                stc1i(ipiv + j0 + c0 + jj, j0 + c0 + bpos);
                if (zero && lds1<3>(sc + 1) == 0) stc1i(sc + 1, j0 + c0 + jj + 1);
            }
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                if (lpos[t] == jj) lpos[t] = bpos;
                else if (lpos[t] == bpos) lpos[t] = jj;
            }
            // ---- multipliers and rank-1 update of the rows below the pivot
            cx<T> uv[kSB];
#pragma unroll
            for (int c = 1; c < kSB; ++c) uv[c] = ldc<3>(u + c);
            const int ncr = sbw - jj;  // columns of the sub-panel from the current one on (uniform)
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                if (lpos[t] > jj && lpos[t] != 0x7fffffff) {
                    const cx<T> l = zero ? x[0][t] : cmul(x[0][t], rp);
                    x[0][t] = l;
#pragma unroll
                    for (int c = 1; c < kSB; ++c)
                        if (c < ncr) cfms(x[c][t], l, uv[c]);  // finished columns sit at the back
                }
            }
            // ---- next column into x[0]; the finished one to the back
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const cx<T> x0 = x[0][t];
#pragma unroll
                for (int c = 0; c + 1 < kSB; ++c) x[c][t] = x[c + 1][t];
                x[kSB - 1][t] = x0;
            }
        }
        // back to x[c] = column c (kSB rotations in all)
        for (int r = sbw; r < kSB; ++r) {
#pragma unroll
            for (int t = 0; t < RM; ++t) {
                const cx<T> x0 = x[0][t];
#pragma unroll
                for (int c = 0; c + 1 < kSB; ++c) x[c][t] = x[c + 1][t];
                x[kSB - 1][t] = x0;
            }
        }
    }
    // the sub-panel at its new rows (every element to a distinct position;
    // nothing reads these columns now) and the list of moved rows
#pragma unroll
    for (int t = 0; t < RM; ++t) {
        const int r = tid + kThreads * t;
        if (r < mq) {
#pragma unroll
            for (int c = 0; c < kSB; ++c)
                if (c < sbw) stc<3>(Q + (lpos[t] + (size_t)c * ldp), x[c][t]);
            if (lpos[t] != r) {
                const int idx = atomicAdd(sc + 12, 1);
                mvl[idx] = make_int2(c0 + r, c0 + lpos[t]);
            }
        }
    }
    subpanel_moves<T>(P, ldp, jbl, c0, sbw, j0, rmap, sc, mvl);
}

// ---- one-wavefront sub-panel (complex64, at most 64 RW rows) --------------------------------
// The same factorisation as subpanel_factor, with every row of the sub-panel
// in wave 0's registers: lane l holds rows l + 64 t (t < RW), x[c][t] =
// column c.  The column loop is unrolled, so no rotation is needed; per column
// the argmax is one DPP reduction (the same packed keys and tie-breaking), the
// winner's lane and register come back uniform, and the pivot row reaches
// every lane by readlane -- no LDS exchange and no barrier per column.  The
// other waves wait at subpanel_moves' first barrier.
template <int RW>
__device__ __forceinline__ void subpanel_factor_1w(cx<float>* __restrict__ P, int m, int ldp, int jbl, int c0, int sbw,
                                                   int j0, int* ipiv, int* rmap, int* sc, int2* mvl) {
    static_assert(RW >= 1 && RW <= 4, "one wavefront holds at most 256 rows");
    const int tid = threadIdx.x;
    const int mq = m - c0;
    cx<float>* Q = P + c0 + (size_t)c0 * ldp;  // sub-panel origin, ld ldp
    if (tid < 64) {
        const int lane = tid;
        cx<float> x[kSB][RW];
        int lpos[RW];  // logical position in the sub-panel; -1: no row
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int r = lane + 64 * t;
            lpos[t] = r < mq ? r : -1;
#pragma unroll
            for (int c = 0; c < kSB; ++c)
                x[c][t] = ldz<3>(Q + (min(r, mq - 1) + (size_t)min(c, sbw - 1) * ldp), c < sbw && r < mq);
        }
        if (lane == 0) stc1i(sc + 12, 0);
        // column jj of the sub-panel; instantiated for jj = 0 .. 15 so that every
        // register index is static
        auto column = [&](auto jc) {
            constexpr int jj = decltype(jc)::value;
            if (jj >= sbw) return;
            unsigned long long pk = 0;
#pragma unroll
            for (int t = 0; t < RW; ++t) {
                const bool elig = lpos[t] >= jj;
                const unsigned long long k =
                    elig ? (pivot_ukey(cabs1(x[jj][t]), lpos[t] == jj) << 20) |
                               ((unsigned)(1023 - lpos[t]) << 10) | (unsigned)(lane + 64 * t)
                         : 0ull;
                pk = k > pk ? k : pk;
            }
            wave_argmax64(pk);
            const unsigned lo = (unsigned)(pk & 0xFFFFFull);
            const int lw = (int)(lo & 63u), tw = (int)((lo >> 6) & 15u);
            const int bpos = 1023 - (int)(lo >> 10);
            // the pivot row, columns jj .. 15, uniform in every lane
            cx<float> uv[kSB];
#pragma unroll
            for (int c = 0; c < kSB; ++c) uv[c] = czero<float>();
#pragma unroll
            for (int t = 0; t < RW; ++t) {
                if (tw == t) {
#pragma unroll
                    for (int c = jj; c < kSB; ++c) {
                        uv[c].re = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[c][t].re), lw));
                        uv[c].im = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[c][t].im), lw));
                    }
                }
            }
            const cx<float> pv = uv[jj];
            const bool zero = pv.re == 0.f && pv.im == 0.f;
            const cx<float> rp = zero ? czero<float>() : crecip(pv);
            if (lane == 0) {
                stc1i(ipiv + j0 + c0 + jj, j0 + c0 + bpos);
                if (zero && lds1<3>(sc + 1) == 0) stc1i(sc + 1, j0 + c0 + jj + 1);
            }
#pragma unroll
            for (int t = 0; t < RW; ++t) {
                if (lpos[t] == jj) lpos[t] = bpos;
                else if (lpos[t] == bpos) lpos[t] = jj;
            }
            // multipliers and rank-1 update of the rows below the pivot
#pragma unroll
            for (int t = 0; t < RW; ++t) {
                if (lpos[t] > jj) {
                    const cx<float> l = zero ? x[jj][t] : cmul(x[jj][t], rp);
                    x[jj][t] = l;
#pragma unroll
                    for (int c = jj + 1; c < kSB; ++c) cfms(x[c][t], l, uv[c]);
                }
            }
        };
        static_for(column, std::make_integer_sequence<int, kSB>{});
        // the sub-panel at its new rows and the list of moved rows
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            const int r = lane + 64 * t;
            if (r < mq) {
#pragma unroll
                for (int c = 0; c < kSB; ++c)
                    if (c < sbw) stc<3>(Q + (lpos[t] + (size_t)c * ldp), x[c][t]);
                if (lpos[t] != r) {
                    const int idx = atomicAdd(sc + 12, 1);
                    mvl[idx] = make_int2(c0 + r, c0 + lpos[t]);
                }
            }
        }
    }
    subpanel_moves<float>(P, ldp, jbl, c0, sbw, j0, rmap, sc, mvl);
}

// ---- inverse of a unit-lower 16 x 16 diagonal block ----------------------------------------
// From Q (LDS, ld ldq; kb <= 16 valid rows/columns), by forward substitution
// X[i][c] -= L[i][k] X[k][c] (i > k) over 256 threads, one entry each;
// X[k][c] comes from the same wavefront by one cross-lane read per part.
// Linv (LDS, 16 x 16, ld 16) is zero outside the kb x kb block; Lg (slot,
// ld kb) gets the kb x kb block for the triangular solves.
template <typename T>
__device__ __forceinline__ void invert_unit_lower16(const cx<T>* Q, int ldq, int kb, cx<T>* Linv,
                                                    cx<T>* __restrict__ Lg) {
    static_assert(kThreads >= kSB * kSB, "one thread per entry of the block");
    const int tid = threadIdx.x;
    if (kThreads > kSB * kSB && tid >= kSB * kSB) return;
    const int i = tid & 15, c = tid >> 4;  // thread (i, c) holds X[i][c]
    cx<T> lrow[kSB - 1];                   // L[i][k] for k < i (zero for rows >= kb)
#pragma unroll
    for (int k = 0; k < kSB - 1; ++k)
        lrow[k] = ldz<3>(Q + (min(i, kb - 1) + (size_t)min(k, kb - 1) * ldq), k < i && i < kb);
    cx<T> x = (i == c && c < kb) ? cmk<T>(T(1), T(0)) : czero<T>();
    static_for([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (k < kb - 1) {
            // X[k][c] sits on lane k + 16 (c % 4) of this wavefront: lane k of the row
            const cx<T> xk = crowbcast<k>(x);
            if (i > k) cfms(x, lrow[k], xk);
        }
    }, std::make_integer_sequence<int, kSB - 1>{});
    stc<3>(Linv + (i + c * kSB), x);
    if (i < kb && c < kb) stc<1>(Lg + (i + (size_t)c * kb), x);
}

// ---- update of the panel's columns right of sub-panel c0 (MFMA, LDS) ------------------------
// Rows [c0, c0+16): U = Linv A (the block row of U); rows [c0+16, m):
// A -= L U.  Columns [c0 + 16, jbl) in chunks of 16.
template <typename T>
__device__ __forceinline__ void inpanel_update(cx<T>* __restrict__ P, int m, int ldp, int jbl, int c0,
                                               const cx<T>* Linv) {
    using M = Mfma<T>;
    using acc_t = typename M::acc;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int cr = c0 + kSB;              // first column (and row) right of / below the block
    const int nchk = (jbl - cr + kSB - 1) / kSB;
    // block row of U, one chunk per wave
    for (int ch = wave; ch < nchk; ch += kWaves) {
        const int cb = cr + kSB * ch, cw = min(kSB, jbl - cb);
        acc_t ure, uim;
        acc_zero<T>(ure);
        acc_zero<T>(uim);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = M::row(lg, s);
            const cx<T> a = ldc<3>(Linv + (li + k * kSB));
            const cx<T> b = ldz<3>(P + ((c0 + k) + (size_t)(cb + min(li, cw - 1)) * ldp), li < cw);
            cmfma<T>(ure, uim, a, b.re, b.im);
        }
        if (li < cw)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                stc<3>(P + ((c0 + M::row(lg, r)) + (size_t)(cb + li) * ldp), cmk<T>(ure[r], uim[r]));
    }
    __syncthreads();
    // rows below: (row tile, chunk) units round-robin over the waves
    const int ntile = (m - cr + kSB - 1) / kSB;
    for (int u = wave; u < ntile * nchk; u += kWaves) {
        const int it = u / nchk, ch = u - it * nchk;
        const int cb = cr + kSB * ch, cw = min(kSB, jbl - cb);
        const int r0 = cr + kSB * it;
        acc_t dre, dim;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + M::row(lg, r);
            const cx<T> v = ldz<3>(P + (min(row, m - 1) + (size_t)(cb + min(li, cw - 1)) * ldp), row < m && li < cw);
            dre[r] = v.re;
            dim[r] = v.im;
        }
        const int arow = min(r0 + li, m - 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = M::row(lg, s);
            cx<T> a = ldc<3>(P + (arow + (size_t)(c0 + k) * ldp));
            a.re = -a.re;
            a.im = -a.im;
            const cx<T> b = ldz<3>(P + ((c0 + k) + (size_t)(cb + min(li, cw - 1)) * ldp), li < cw);
            cmfma<T>(dre, dim, a, b.re, b.im);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + M::row(lg, r);
            if (row < m && li < cw) stc<3>(P + (row + (size_t)(cb + li) * ldp), cmk<T>(dre[r], dim[r]));
        }
    }
    __syncthreads();
}

// ---- left-looking update of the next columns -------------------------------------------------
// Columns [j0, j0 + wl) of the factorisation, wl <= 16 NCT, brought up to date with
// the finished 16-column blocks b = kb0 .. kb1-1: with A the columns (rows in
// logical order), per block U_b = Linv_b A_b (its block row), then A_t -= L_tb U_b for
// the row tiles t > b.  The columns stay in the accumulators throughout: row tiles are dealt to
// the wavefronts (tile kWaves q + wave), a tile's register r of lane li + 16 lg
// holds row M::row(lg, r), column li.  L_tb is read from the slot straight into MFMA operands,
// one group of tiles ahead of its use (it does not depend on the chain of
// the U_b); U_b goes through LDS (ub, two alternating buffers) to every wavefront and to the
// slot.  The owner of tile b + 1 updates it first and forms U_{b+1} before its other
// tiles, so one barrier per block carries the chain.
//
// Each entry of L is read once per 16 NCT columns and each entry of the matrix is written
// once.  The right-looking update that this replaces read and wrote the whole
// trailing matrix per LDS panel (n = 256: 10.2 against 3.5 MB a point in complex128,
// 4.4 of 5.2 TB/s, its bound).
//
// from_slot: the columns' current values are in the slot (partly updated), else A(w) is
// assembled from the operators; right-hand sides (columns from n on) are in the slot.  Afterwards the rows
// from kb1 * 16 on go to the LDS panel P (ld ldp, the first wp columns, padded with zeros
// to a multiple of 16) and to the slot (the columns from wp on).
// G3: Gauss 3M products (three accumulators, converted at the ends and every 32 finished
// columns: x and y grow with the columns and cancel in z - x - y.  Converted at the ends only,
// the factors were 8 % less exact, 41 % at worst, n = 256; the conversions cost 2 %.  Four
// products take as long as that (n = 129..256: 0.98..1.01) and make factors 11 % more exact,
// but refined solutions near resonances are less so: at tol 1e-15 the 99.9th percentile of
// the error against the closed form was 2e-11..1.1e-10, with three 1.1e-11..2e-11.)
constexpr int kPB = 8;  // panel columns loaded per batch

template <typename T, int MAXR, int NCT, bool G3>
__device__ __forceinline__ void left_update(const SysDesc& sd, double w, double w2, cx<T>* __restrict__ S,
                                            const cx<T>* __restrict__ Lg, int n, const int* rmap, int j0, int wl,
                                            int kb0, int kb1, bool from_slot, bool whole, cx<T>* P, int ldp, int wp) {
    using M = Mfma<T>;
    using acc_t = typename M::acc;
    constexpr int NRT = 4 * MAXR / kWaves;       // row tiles per wavefront
    constexpr int NR = NRT < 4 ? NRT : 4;        // operand buffers: L is loaded NR tiles ahead
    constexpr int UL = 17;                       // leading dimension of a U block in LDS
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int ntile = (n + kSB - 1) / kSB;
    cx<T>* ub = P;  // the panel region and what follows it are free until the end
    int plr[NRT];   // physical row of row li of each tile
    acc_t cr[NRT][NCT], ci[NRT][NCT], cy[G3 ? NRT : 1][NCT];
    // ---- the first operands of the blocks, in flight while the columns are read
#pragma unroll
    for (int q = 0; q < NRT; ++q) plr[q] = lds1<3>(rmap + min(kSB * (wave + kWaves * q) + li, n - 1));
    cx<T> lb[NR][4];  // L_tb operands: [buffer][k-step]
    auto load_l = [&](int b, int q, int pr, cx<T> (&l)[4]) {
        const int t = wave + kWaves * q;
        if (t > b && t < ntile)
#pragma unroll
            for (int k = 0; k < 4; ++k) l[k] = ldc<1>(S + (pr + (size_t)(kSB * b + M::row(lg, k)) * n));
    };
    // the inverted diagonal block of this wavefront's next tile in the chain; zero beyond a
    // narrow last block (stored with its own width as leading dimension)
    cx<T> linv[4];
    int tl = wave;
    while (tl < kb0) tl += kWaves;
    auto load_linv = [&]() {
        if (tl < kb1) {
            const int kb = min(kSB, n - kSB * tl);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int kk = M::row(lg, k);
                linv[k] = ldz<1>(Lg + ((size_t)tl * kSB * kSB + min(li, kb - 1) + min(kk, kb - 1) * kb), li < kb && kk < kb);
            }
        }
    };
    if (kb1 > kb0) {
        load_linv();
#pragma unroll
        for (int q = 0; q < NR; ++q) load_l(kb0, q, plr[q], lb[q]);
    }
    // ---- the columns as they stand, read along the rows (coalesced) into LDS, all at
    // once where the region holds them (whole), else 16 at a time, and from there into the tiles
    const int ldn = n | 1, rb = kSB * kb0, nr = n - rb;
    static_for([&](auto cc) {
        constexpr int c = decltype(cc)::value;
#pragma unroll
        for (int q = 0; q < NRT; ++q) {
            acc_zero<T>(cr[q][c]);
            acc_zero<T>(ci[q][c]);
        }
        if (kSB * c < wl) {
            if (c == 0 || !whole) {
                const int nc = min(whole ? kSB * NCT : kSB, wl - kSB * c);
                const int na = from_slot ? 0 : max(0, min(nc, n - j0 - kSB * c));  // assembled
                auto fill = [&](int c0, int c1, auto&& entry) {
                    const int nbat = (c1 - c0 + kPB - 1) / kPB;
                    for (int e = tid; e < nr * nbat; e += kThreads) {
                        const int r = rb + e % nr, cb = c0 + e / nr * kPB;
                        const int pr = lds1<3>(rmap + r);
                        cx<T> v[kPB];
#pragma unroll
                        for (int u = 0; u < kPB; ++u) v[u] = entry(pr + (size_t)(j0 + kSB * c + min(cb + u, c1 - 1)) * n);
#pragma unroll
                        for (int u = 0; u < kPB; ++u)
                            if (cb + u < c1) stc<3>(P + (r + (cb + u) * ldn), v[u]);
                    }
                };
                if (c) __syncthreads();
                if (na < nc) fill(na, nc, [&](size_t e) { return ldc<1>(S + e); });
                if (na > 0)
                    with_kind(sd, [&](auto kc) { fill(0, na, [&](size_t e) { return to_t<T>(elem_at<decltype(kc)::value>(sd, e, w, w2)); }); });
                __syncthreads();
            }
            const cx<T>* pt = P + (whole ? kSB * c * ldn : 0);
#pragma unroll
            for (int q = 0; q < NRT; ++q) {
                const int t = wave + kWaves * q;
                if (t < ntile && t >= kb0)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const cx<T> v = ldc<3>(pt + (min(kSB * t + M::row(lg, r), n - 1) + min(li, wl - kSB * c - 1) * ldn));
                        cr[q][c][r] = v.re;
                        ci[q][c][r] = v.im;
                    }
            }
        }
    }, std::make_integer_sequence<int, NCT>{});
    __syncthreads();  // the region's next use: U blocks, or the panel
    if (kb1 > kb0) {
        // Gauss form: x = cr (starts at d_r), y = cy (0), z = ci (d_r + d_i)
        auto to_gauss = [&](int q, int c) {
            acc_zero<T>(cy[G3 ? q : 0][c]);
#pragma unroll
            for (int r = 0; r < 4; ++r) ci[q][c][r] += cr[q][c][r];
        };
        auto from_gauss = [&](int q, int c) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const T x = cr[q][c][r], y = cy[G3 ? q : 0][c][r];
                cr[q][c][r] = x - y;
                // an infinite real part would leave NaN: z - x
                ci[q][c][r] = fabs(x) == T(__builtin_inf()) ? T(0) : ci[q][c][r] - x - y;
            }
        };
        if (G3)
#pragma unroll
            for (int q = 0; q < NRT; ++q)
#pragma unroll
                for (int c = 0; c < NCT; ++c) to_gauss(q, c);
        // U_t = Linv_t A_t of tile q into its LDS buffer
        auto make_u = [&](auto qc) {
            constexpr int q = decltype(qc)::value;
            cx<T>* u = ub + (tl & 1) * NCT * kSB * UL;
#pragma unroll
            for (int c = 0; c < NCT; ++c) {
                if (G3) from_gauss(q, c);
                acc_t ur, ui;
                acc_zero<T>(ur);
                acc_zero<T>(ui);
#pragma unroll
                for (int k = 0; k < 4; ++k) cmfma<T>(ur, ui, linv[k], cr[q][c][k], ci[q][c][k]);
#pragma unroll
                for (int r = 0; r < 4; ++r) stc<3>(u + ((kSB * c + li) * UL + M::row(lg, r)), cmk<T>(ur[r], ui[r]));
            }
            tl += kWaves;
            load_linv();
        };
        static_for([&](auto qc) {
            if (wave + kWaves * decltype(qc)::value == kb0) make_u(qc);
        }, std::make_integer_sequence<int, NRT>{});
        __syncthreads();
        for (int b = kb0; b < kb1; ++b) {
            const cx<T>* u = ub + (b & 1) * NCT * kSB * UL;
            T vr[NCT][4], vi[NCT][4];
#pragma unroll
            for (int c = 0; c < NCT; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const cx<T> v = ldc<3>(u + ((kSB * c + li) * UL + M::row(lg, k)));
                    vr[c][k] = v.re;
                    vi[c][k] = v.im;
                }
            // U_b to the slot, 16 rows of a column together
            for (int e = tid; e < kSB * wl; e += kThreads) {
                const int r = e & (kSB - 1), c = e / kSB;
                if (kSB * b + r < n)
                    stc<1>(S + (lds1<3>(rmap + kSB * b + r) + (size_t)(j0 + c) * n), ldc<3>(u + (c * UL + r)));
            }
            static_for([&](auto qc) {
                constexpr int q = decltype(qc)::value, lq = (q + NR) % NRT;
                const int t = wave + kWaves * q;
                if (t > b && t < ntile) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const cx<T> l = cmk<T>(-lb[q % NR][k].re, -lb[q % NR][k].im);
                        if (G3) {
                            const T ls = l.re + l.im;
#pragma unroll
                            for (int c = 0; c < NCT; ++c)
                                cmfma3<T>(cr[q][c], cy[G3 ? q : 0][c], ci[q][c], l, ls, vr[c][k], vi[c][k]);
                        } else {
#pragma unroll
                            for (int c = 0; c < NCT; ++c) cmfma<T>(cr[q][c], ci[q][c], l, vr[c][k], vi[c][k]);
                        }
                    }
                }
                // the buffer's next use: NR tiles on, of this block or the next
                const int bn = q + NR < NRT ? b : b + 1;
                if (bn < kb1) load_l(bn, lq, plr[lq], lb[q % NR]);
                if (t == b + 1 && t < ntile && b + 1 < kb1) make_u(qc);
                else if (G3 && (b - kb0) % 2 && b + 1 < kb1 && t > b && t < ntile)
#pragma unroll
                    for (int c = 0; c < NCT; ++c) {
                        from_gauss(q, c);
                        to_gauss(q, c);
                    }
            }, std::make_integer_sequence<int, NRT>{});
            __syncthreads();
        }
        if (G3)
#pragma unroll
            for (int q = 0; q < NRT; ++q)
                if (wave + kWaves * q >= kb1)
#pragma unroll
                    for (int c = 0; c < NCT; ++c) from_gauss(q, c);
    }
    // ---- the updated rows to the LDS panel and to the slot
    const int r0 = kSB * kb1;
#pragma unroll
    for (int q = 0; q < NRT; ++q) {
        const int t = wave + kWaves * q;
        if (t >= kb1 && t < ntile) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = kSB * t + M::row(lg, r);
                if (row < n) {
                    const int pr = lds1<3>(rmap + row);
#pragma unroll
                    for (int c = 0; c < NCT; ++c) {
                        const int cc = kSB * c + li;
                        const cx<T> v = cmk<T>(cr[q][c][r], ci[q][c][r]);
                        if (kSB * c < wp) stc<3>(P + (row - r0 + (size_t)cc * ldp), cc < wp ? v : czero<T>());
                        if (cc >= wp && cc < wl) stc<1>(S + (pr + (size_t)(j0 + cc) * n), v);
                    }
                }
            }
        }
    }
}

// ---- the wide-panel factorisation ------------------------------------------------------------
// Left-looking in steps of 16 NCT columns (32 complex64, 16 complex128: what the
// accumulators hold beside the operands), each step one or two LDS panels of jb columns; the
// first group of right-hand sides last, as columns n .. n + nr - 1.  Where the last step has
// room for them they are its columns too, and only its own blocks are left to apply
// afterwards (a pass over all blocks for them alone made n = 129..132 plain 2 to 4 % slower than
// right-looking panels had been: n = 129, 1 load, 1024 points 846 us, 795 now).
template <typename T, int MAXR, bool G3>
__device__ __forceinline__ void factor_wide(const SysDesc& s, double w, double w2, cx<T>* __restrict__ S,
                                            const Layout& lay, const Lds& L, int nr) {
    constexpr int NCT = sizeof(T) == 4 ? 2 : 1;
    constexpr int W = kSB * NCT;
    const int n = s.n, tid = threadIdx.x;
    const size_t nn = (size_t)n * n;
    const int jb = lay.jb;
    char* base = L.main;
    cx<T>* P = reinterpret_cast<cx<T>*>(base);
    base += align16((long long)(n | 1) * jb * sizeof(cx<T>));
    cx<T>* Linv = reinterpret_cast<cx<T>*>(base);
    cx<T>* cand = Linv;  // a sub-panel's pivot candidates, read before any of its blocks is inverted
    base += wide_blocks_bytes(jb, (int)sizeof(cx<T>), kWaves);
    int2* mvl = reinterpret_cast<int2*>(base);
    const size_t nblk = (size_t)((n + kSB - 1) / kSB);
    cx<T>* Lg = S + (size_t)n * (n + kMaxGroup);
    cx<T>* Ug = Lg + nblk * kSB * kSB;

    // right-hand sides eliminated along with the factorisation (columns n .. n+nr-1)
    for (int e = tid; e < n * nr; e += kThreads) {
        const int r = e % n, g = e / n;
        stc<1>(S + (nn + (size_t)g * n + r),
               to_t<T>(ldc<1>(reinterpret_cast<const z64*>(s.F) + r + (size_t)g * s.ldf)));
    }
    for (int r = tid; r < n; r += kThreads) L.rmap[r] = r;
    if (tid == 0) L.sc[1] = 0;
    __syncthreads();

    const bool fuse = nr > 0 && (n - 1) % W + 1 + nr <= W;  // room for the right-hand sides
    int jlast = 0;                                          // the last panel's first column
    for (int j0 = 0; j0 < n + (nr > 0 ? 1 : 0);) {
        const bool rhs = j0 >= n;
        const int first = j0 / W * W;  // the step's first column
        const bool cont = !rhs && j0 > first;  // a later panel of the step
        const int jend = rhs || (fuse && first + W >= n) ? n + nr : min(first + W, n);
        const int jbl = rhs ? 0 : min(jb, min(first + W, n) - j0), m = n - j0;
        // complex64: odd leading dimension, so the columns an MFMA operand read
        // spans start in different LDS banks (complex128 elements spread already)
        const int ldp = sizeof(T) == 4 ? (m | 1) : m;
        const int kb0 = cont ? (j0 - jb) / kSB : rhs && fuse ? jlast / kSB : 0;
        left_update<T, MAXR, NCT, G3>(s, w, w2, S, Lg, n, L.rmap, j0, jend - j0, kb0,
                                      rhs ? (int)nblk : j0 / kSB, rhs || cont, jb >= W, P, ldp, jbl);
        __syncthreads();
        if (rhs) break;
        // ---- sub-panels
        for (int c0 = 0; c0 < jbl; c0 += kSB) {
            const int sbw = min(kSB, jbl - c0);
            // the sub-panel's chain of barriers is latency-bound: its waves
            // take issue priority over the other workgroup's update on the CU
            // (complex64: +0.6 %; complex128 measured -0.6 % and keeps 0)
            if (sizeof(T) == 4) __builtin_amdgcn_s_setprio(2);
            // complex64 sub-panels of at most 64 rows: one wavefront, no
            // barrier per column (measured at n = 256: +2.3 %; with up to 256
            // rows in one wavefront its serial rank-1 updates cost about what
            // the barriers save)
            bool one_wave = false;
            if constexpr (sizeof(T) == 4) {
                one_wave = m - c0 <= 64;
                if (one_wave) subpanel_factor_1w<1>(P, m, ldp, jbl, c0, sbw, j0, L.ipiv, L.rmap, L.sc, mvl);
            }
            if (!one_wave) subpanel_factor<T, MAXR>(P, m, ldp, jbl, c0, sbw, j0, L.ipiv, L.rmap, L.sc, cand, mvl);
            if (sizeof(T) == 4) __builtin_amdgcn_s_setprio(0);
            invert_unit_lower16<T>(P + c0 + (size_t)c0 * ldp, ldp, sbw, Linv + (size_t)(c0 / kSB) * kSB * kSB,
                                   Lg + (size_t)((j0 + c0) / kSB) * kSB * kSB);
            __syncthreads();
            if (c0 + kSB < jbl) inpanel_update<T>(P, m, ldp, jbl, c0, Linv + (size_t)(c0 / kSB) * kSB * kSB);
        }
        // ---- the factored panel to the slot (rows at their physical positions)
        for (int r = tid; r < m; r += kThreads) {
            const int pr = lds1<3>(L.rmap + j0 + r);
            for (int c = 0; c < jbl; ++c) stc<1>(S + (pr + (size_t)(j0 + c) * n), ldc<3>(P + (r + (size_t)c * ldp)));
        }
        __syncthreads();
        jlast = j0;
        j0 += jbl;
    }
    if (sizeof(T) == 4) {
        uinv_blocks(S, n, L.rmap, kSB, Ug);
        __syncthreads();
    }
}

}  // namespace stc
