// Grid edges with a two-factor register transform, n = N1*N2 with both factors from the
// small DFTs of fft_reg.h (at most 16): of the even lengths that the reference's factorisation
// rule accepts (2^k with at most 3^2, 5, 7 and 11, Basis.cc:126-154) those from 18 to 256 except
// 22, 198, 220 and 252, and of the longer products of 2, 3 and 5 also 50, 54, 100, 108 and 150.
// All others take the LDS Stockham passes, which make one LDS round trip per radix instead of
// three per transform pair: at 88^3 (108 Al atoms, 195 bands, FP64, MI355X) the x pass took 1.37
// ms and the y passes 0.30 / 0.26 ms per Hψ on Stockham passes, and a two-cycle SCF 41.1 ms
// against 28.6 ms on the register ones.
// FP32 takes the same transforms at the E lengths.  At the D lengths (FP64 only) its factors are
// those of F, whose transform keeps the radix order, tabled twiddles and so the rounding of the
// Stockham passes that FP32 ran on there (stockham_order): its first factor is the product of
// the leading radices of the Stockham plan, the second the last radix.  The repeated products
// of the E form cost FP32 accuracy (Hψ at 110^3: error 2.7e-8 against 2.2e-8 of the result); F
// forms return the Stockham results bit for bit.  The passes of a local FP32 Hψ (MI355X,
// before -> after): 56^3, 64 bands 0.21 -> 0.07 ms; 88^3, 195 bands 1.21 -> 0.55 ms; 110^3, 300
// bands 3.04 -> 1.31 ms; 112^3, 512 bands 5.28 -> 2.50 ms.
// FP32 at 126 and 150, whose plans have no such split, keeps the Stockham passes.
// Each QBH_EDGES_<p> is one compilation unit (qbh_fft_edges.hip with QBH_FFT_PART = p), the
// lengths dealt so that the units take about the same time to compile.
#pragma once

#define QBH_EDGES_0(E, D, F) D(6, 3) F(6, 3) E(9, 6) E(10, 9) E(14, 10)
#define QBH_EDGES_1(E, D, F) D(5, 4) F(4, 5) D(8, 7) F(8, 7) E(12, 8) E(12, 12)
#define QBH_EDGES_2(E, D, F) D(6, 4) F(8, 3) E(10, 6) E(10, 10) D(15, 10)
#define QBH_EDGES_3(E, D, F) E(7, 4) E(8, 8) E(12, 9) D(14, 11) F(14, 11)
#define QBH_EDGES_4(E, D, F) D(6, 5) F(6, 5) D(11, 6) F(6, 11) D(11, 10) F(10, 11) E(16, 10)
#define QBH_EDGES_5(E, D, F) E(8, 4) D(10, 7) F(10, 7) D(14, 8) F(16, 7) E(14, 12)
#define QBH_EDGES_6(E, D, F) E(6, 6) E(9, 8) E(12, 10) D(16, 11) F(16, 11)
#define QBH_EDGES_7(E, D, F) E(8, 5) E(10, 8) D(14, 9) E(15, 12)
#define QBH_EDGES_8(E, D, F) D(7, 6) F(6, 7) D(12, 7) F(12, 7) E(16, 8) E(16, 12)
#define QBH_EDGES_9(E, D, F) D(11, 4) F(4, 11) E(8, 6) D(11, 8) F(8, 11) D(12, 11) F(12, 11) E(15, 14)
#define QBH_EDGES_10(E, D, F) E(10, 5) E(16, 14) E(16, 15)
#define QBH_EDGES_11(E, D, F) E(16, 16)
#define QBH_EDGE_PARTS(P) P(0) P(1) P(2) P(3) P(4) P(5) P(6) P(7) P(8) P(9) P(10) P(11)

#define QBH_EDGE_IS(N1, N2) || n == (N1) * (N2)
#define QBH_EDGE_SKIP(N1, N2)
#define QBH_EDGE_IN(p) QBH_EDGES_##p(QBH_EDGE_SKIP, QBH_EDGE_SKIP, QBH_EDGE_IS)
// whether the FP32 transform of edge n is an F form
constexpr bool stockham_length(int n) { return false QBH_EDGE_PARTS(QBH_EDGE_IN); }
