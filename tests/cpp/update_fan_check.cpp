// update_fan_f64 against update_ref_f64_x, bit for bit (NaN equals NaN): random
// triangles of many shapes and scales, and arrival times of a plane wave (also
// along an edge, where a condition is 0 up to rounding), a point, equal, random.
// Prints the triangles compared and how many took the conditions in full.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../gproshan_amd/csrc/update_step.hpp"

using namespace gp;

int main(int argc, char **argv)
{
	const long n = argc > 1 ? atol(argv[1]) : 1000000;
	std::mt19937_64 g(argc > 2 ? atol(argv[2]) : 1);
	std::normal_distribution<double> N;
	std::uniform_real_distribution<double> U(-1, 1);
	long bad = 0, planar = 0, nan = 0;
	for (long k = 0; k < n; k++) {
		double X0[3], X1[3];
		const int shape = g() % 6;
		const double scale = std::ldexp(1 + std::abs(U(g)), (int) (g() % 7 == 0 ? (long) (g() % 180) - 90 : (long) (g() % 9) - 8));
		for (int c = 0; c < 3; c++) { X0[c] = N(g); X1[c] = N(g); }
		if (shape == 0) { X0[2] = X1[2] = 0; for (int c = 0; c < 2; c++) { X0[c] = (int) (g() % 5) - 2; X1[c] = (int) (g() % 5) - 2; } }
		if (shape == 1) for (int c = 0; c < 3; c++) X1[c] = X0[c] * (1 + U(g)) + std::ldexp(N(g), -(int) (g() % 50));
		if (shape == 2) { const double f = std::ldexp(1, (int) (g() % 40) - 20); for (double &x : X1) x *= f; }
		if (shape == 3) { X0[1] = X0[2] = 0; X1[0] = std::ldexp(X1[0], -(int) (g() % 60)); X1[2] = 0; }
		for (int c = 0; c < 3; c++) { X0[c] *= scale; X1[c] *= scale; }
		if (!fan_vector(X0) || !fan_vector(X1)) { k--; continue; }
		const double l0 = std::sqrt(ref_sq(X0)), l1 = std::sqrt(ref_sq(X1));
		double t0 = 0, t1 = 0;
		const double base = g() % 4 ? std::abs(N(g)) * 100 * scale : 0;
		switch (g() % 7) {
		case 0: t0 = base + l0 * std::abs(N(g)); t1 = base + l1 * std::abs(N(g)); break;
		case 1: { double w[3] = { U(g), U(g), U(g) }; const double m = std::sqrt(ref_sq(w));
			t0 = base + 10 * scale; t1 = t0; for (int c = 0; c < 3; c++) { t0 += X0[c] * w[c] / m; t1 += X1[c] * w[c] / m; } break; }
		case 2: t0 = t1 = base; break;
		case 3: { double s[3], a[3], b[3]; for (int c = 0; c < 3; c++) { s[c] = N(g) * 5 * scale; a[c] = X0[c] - s[c]; b[c] = X1[c] - s[c]; }
			t0 = std::sqrt(ref_sq(a)); t1 = std::sqrt(ref_sq(b)); break; }
		case 4: { const double d = X0[0] * X1[0] + X0[1] * X1[1] + X0[2] * X1[2];   // the front runs along an edge
			t0 = base + 3 * scale; t1 = g() & 1 ? t0 - l0 + d / l0 : t0 + l0 - d / l0; break; }
		case 5: t0 = g() & 1 ? INFINITY : base; t1 = g() & 1 ? INFINITY : base; break;
		default: t0 = base; t1 = g() & 1 ? base + l1 : 0;
		}
		if (!(t0 >= 0)) t0 = 0;
		if (!(t1 >= 0)) t1 = 0;
		const double a = update_ref_f64_x(X0, X1, t0, t1);
		const double b = update_fan_f64(X0, X1, ref_sq(X0), ref_sq(X1), fan_sqrt(ref_sq(X0)), fan_sqrt(ref_sq(X1)), t0, t1);
		if (a != a) nan++;
		else if (a != t0 + l0 && a != t1 + l1) planar++;
		if (std::memcmp(&a, &b, 8) != 0 && !(a != a && b != b)) {
			if (bad++ < 5) std::printf("%a %a %a  %a %a %a  %a %a: %a %a\n", X0[0], X0[1], X0[2], X1[0], X1[1], X1[2], t0, t1, a, b);
		}
	}
	std::printf("%ld triangles, %ld planar, %ld NaN, %ld differ\n", n, planar, nan, bad);
	return bad != 0;
}
