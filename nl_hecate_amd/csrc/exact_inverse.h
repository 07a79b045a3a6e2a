// Text of the chunk inverse inside the kernels of exact_mm.hip, included once per direction (as functions the same code
// compiled to 7 us more of a 250 us kernel: conditions on the wave index became vector compares).
// T = (I - Lam)^-1 for the unit lower triangular system of a chunk, by blocks of 16 tokens.  INV_L: Lam (overwritten),
// INV_D: the diagonal blocks' inverses, INV_N: N = D Lam_off, then T, INV_X: scratch (all in LDS); INV_BESIDE_N: what
// else runs beside the product for N; INV_OUT(row, col, x): what else happens to T's elements.  A barrier stands before
// (Lam complete) and after.  Needs w, l, ib, m0 and MMAT of the kernel.
    if (w < 4 && l < 16) {
        // D_b = (I - Lam_bb)^-1 by substitution: lane c holds column c of block b = w
        const float *A = INV_L + (16 * w) * LDM + 16 * w;
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            float acc = r == l ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < r; j++) acc = fmaf(A[r * LDM + j], x[j], acc);
            x[r] = acc;
        }
        float *Dd = INV_D + (16 * w) * LDM + 16 * w + l;
#pragma unroll
        for (int r = 0; r < 16; r++) Dd[r * LDM] = x[r];
    }
    __syncthreads();
    {   // N = D Lam_off
#pragma unroll
        for (int tl = 0; tl < 2; tl++) {
            const int jb = 2 * (w & 1) + tl;
            f32x4 nacc = {0.f, 0.f, 0.f, 0.f};
            if (jb < ib)
                MMAT(nacc, [&](int m, int kk) { return INV_D[(m0 + m) * LDM + kk]; },
                           [&](int kk, int n) { return INV_L[kk * LDM + 16 * jb + n]; }, 16 * ib);
#pragma unroll
            for (int i = 0; i < 4; i++) INV_N[(m0 + row_of(i, l)) * LDM + 16 * jb + (l & 15)] = nacc[i];
        }
        INV_BESIDE_N
    }
    __syncthreads();
    auto aN = [&](int m, int kk) { return INV_N[(m0 + m) * LDM + kk]; };
    // N is strictly block lower triangular (blocks of 16): its powers need only the block products that can be non-zero
#pragma unroll
    for (int tl = 0; tl < 2; tl++) {   // N^2 -> Lam's place
        const int jb = 2 * (w & 1) + tl;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = jb + 1; kb < ib; kb++)
            MMAT(acc, aN, [&](int kk, int n) { return INV_N[kk * LDM + 16 * jb + n]; }, 16 * kb);
#pragma unroll
        for (int i = 0; i < 4; i++) INV_L[(m0 + row_of(i, l)) * LDM + 16 * jb + (l & 15)] = acc[i];
    }
    __syncthreads();
#pragma unroll
    for (int tl = 0; tl < 2; tl++) {   // X = (I + N)(I + N^2) = I + N + N^2 + N N^2
        const int jb = 2 * (w & 1) + tl;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = jb + 2; kb < ib; kb++)
            MMAT(acc, aN, [&](int kk, int n) { return INV_L[kk * LDM + 16 * jb + n]; }, 16 * kb);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = m0 + row_of(i, l), col = 16 * jb + (l & 15);
            INV_X[row * LDM + col] = acc[i] + INV_N[row * LDM + col] + INV_L[row * LDM + col] + (row == col ? 1.f : 0.f);
        }
    }
    __syncthreads();
    {   // T = X D
#pragma unroll
        for (int tl = 0; tl < 2; tl++) {
            const int jb = 2 * (w & 1) + tl;
            f32x4 t = {0.f, 0.f, 0.f, 0.f};
            MMAT(t, [&](int m, int kk) { return INV_X[(m0 + m) * LDM + kk]; },
                       [&](int kk, int n) { return INV_D[kk * LDM + 16 * jb + n]; }, 16 * jb);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = 16 * jb + (l & 15);
                INV_N[row * LDM + col] = t[i];
                INV_OUT(row, col, t[i])
            }
        }
    }
    __syncthreads();
#undef INV_L
#undef INV_D
#undef INV_N
#undef INV_X
#undef INV_BESIDE_N
#undef INV_OUT
