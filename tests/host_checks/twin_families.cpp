// A table with two order-2 irreps of one l loads, with the order-3 families left to
// the kernels that add any number of families to a row; the table as it is takes the
// order-3 kernel.  Arguments: the table's text, a folder for the potential files.
#include <cstdio>
#include <fstream>
#include <sstream>
#include <string>

#include "model.h"

extern "C" {
extern const char mlip_gtinv_table_begin[1] = {0};
extern const char mlip_gtinv_table_end[1] = {0};
}

using namespace mlip;

static void write(const std::string& path, int n) {
    std::ofstream f(path);
    f << "Ti Al # element\n5.0 # cutoff\ngaussian # pair_type\ngtinv # des_type\n4 # model_type\n1 # max_p\n"
         "4 # max_l\n3 # gtinv_order\n4 4 # gtinv_maxl\n0 0 # gtinv_sym\n"
      << n << " # n\n";
    for (int line = 0; line < 2; ++line)
        for (int k = 0; k < n; ++k) f << "1.0" << (k + 1 < n ? " " : "\n");
    f << "2 # number of parameters\n1.0 0.0 # pair func. params\n1.0 2.0 # pair func. params\n30.0 30.0 # mass\n";
}

static bool load(const GtinvTable& table, const std::string& folder, Model& m) {
    const std::string path = folder + "/p.mlip";
    std::string err;
    Model probe;
    write(path, 1);
    if (!load_model(path, table, probe, err, false)) return std::printf("%s\n", err.c_str()), false;
    write(path, probe.n_coeff);
    if (!load_model(path, table, m, err)) return std::printf("%s\n", err.c_str()), false;
    return true;
}

int main(int, char** argv) {
    std::ifstream in(argv[1]);
    std::stringstream text;
    text << in.rdbuf();
    GtinvTable table;
    std::string err;
    if (!parse_gtinv_text(text.str().data(), text.str().size(), table, err)) return std::printf("%s\n", err.c_str()), 1;
    Model plain, twins;
    if (!load(table, argv[2], plain)) return 1;
    size_t at = 0;
    while (table.irreps[at].l.size() != 2 || table.irreps[at].l[0] != 2) ++at;
    table.irreps.insert(table.irreps.begin() + static_cast<long>(at), table.irreps[at]);
    if (!load(table, argv[2], twins)) return 1;
    bool order3 = false;
    for (const PlanVisit& q : twins.types[0].plan_adj) order3 = order3 || q.v.order == 3;
    std::printf("order-3 kernel's l: %d, with twins %d\n", plain.lmaxq3, twins.lmaxq3);
    return plain.lmaxq3 == 4 && twins.lmaxq3 == -1 && order3 && twins.n_gtinv > plain.n_gtinv ? 0 : 1;
}
