// Generated by gen_obc_farfield.py -- do not edit by hand.
// Far-field OBC2 pair integral polynomials in y = (s/r)^2 on [0, 0.25].
// max relative error: h 3.13e-08, k 1.24e-08
#pragma once
#define PRX_OBC_FAR_YMAX 0.25f
#define PRX_OBC_FAR_XMAX 0.5f
constexpr int kObcHDeg = 6;
__device__ constexpr double kObcH[7] = {0.66666666666666663, 0.79999510665847684, 0.85752043664690591, 0.8793244578024505, 1.0182343314637758, 0.31617928533729833, 2.4493636164745931};
constexpr int kObcKDeg = 7;
__device__ constexpr double kObcK[8] = {1.3333333333333333, 2.4000048296751366, 3.4280749247723237, 4.4614754950161277, 5.1820909506110944, 8.7370190497025035, -2.5286160932569119, 28.878675143138228};
// The same on [0, 0.0625] (s <= r/4); max relative error: h 4.36e-09, k 1.31e-08
#define PRX_OBC_FAR4_YMAX 0.0625f
#define PRX_OBC_FAR4_XMAX 0.25f
constexpr int kObcH4Deg = 4;
__device__ constexpr double kObcH4[5] = {0.66666666666666663, 0.79999885342697763, 0.85732018962125545, 0.88043463587107751, 1.0650812122317668};
constexpr int kObcK4Deg = 4;
__device__ constexpr double kObcK4[5] = {1.3333333333333333, 2.3999918665486706, 3.429832630543606, 4.3842881074745668, 6.56155401950405};
// The same for s <= r/6.5; max relative error: h 4.74e-09, k 1.28e-08
#define PRX_OBC_FAR3_XMAX 0.153846154f
constexpr int kObcH3Deg = 3, kObcK3Deg = 3;
__device__ constexpr double kObcH3[4] = {0.66666666666666663, 0.8000023143791587, 0.8565514797781687, 0.9315788084603891};
__device__ constexpr double kObcK3[4] = {1.3333333333333333, 2.4000139555160245, 3.4250031263590128, 4.7018282471307984};
// The same for s <= r/14.5; max relative error: h 5.60e-09, k 1.40e-08
#define PRX_OBC_FAR2_XMAX 0.0689655172f
constexpr int kObcH2Deg = 2, kObcK2Deg = 2;
__device__ constexpr double kObcH2[3] = {0.66666666666666663, 0.79999128025053479, 0.86305998163217301};
__device__ constexpr double kObcK2[3] = {1.3333333333333333, 2.3999563587238897, 3.4581841118787842};
