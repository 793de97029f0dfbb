// Prints the choices of csrc/qob_rules.h, one a line, for the questions on
// stdin ("name arguments"); test_rules_host.py compares them.
#include "../quantumopticsbase.jl_amd/csrc/qob_rules.h"

#include <iostream>
#include <sstream>
#include <string>

int main() {
    std::string line, name;
    while (std::getline(std::cin, line)) {
        std::istringstream s(line);
        s >> name;
        if (name == "zgemv_in_one") {
            long long m, n;
            s >> m >> n;
            std::cout << qob::zgemv_in_one(m, n) << "\n";
        } else if (name == "zgemv_t_form") {
            long long c64, k, m;
            s >> c64 >> k >> m;
            const qob::GemvT f = qob::zgemv_t_form(c64 != 0, k, m);
            std::cout << 10 * f.loads + f.elems << "\n";
        } else if (name == "qubit_state_tbits") {
            long long nbits, c64, ncols, two;
            s >> nbits >> c64 >> ncols >> two;
            std::cout << qob::qubit_state_tbits((int)nbits, c64 != 0, ncols, two != 0) << "\n";
        } else if (name == "any_rows") {
            long long c64, n1, P, n3, ncu;
            s >> c64 >> n1 >> P >> n3 >> ncu;
            std::cout << qob::any_rows(c64 != 0, n1, P, n3, ncu) << "\n";
        } else if (name == "one_factor_by_mode") {
            long long c64, total, n1, d;
            s >> c64 >> total >> n1 >> d;
            std::cout << qob::one_factor_by_mode(c64 != 0, total, n1, (int)d) << "\n";
        } else if (name == "group_too_thin") {
            long long c64, n1, W, P, modes;
            s >> c64 >> n1 >> W >> P >> modes;
            std::cout << qob::group_too_thin(c64 != 0, n1, (int)W, P, (int)modes) << "\n";
        } else {
            return 1;
        }
        if (!s) return 2;
    }
    return 0;
}
