cd /root/repo
/usr/local/graft/bin/gpurun --timeout 300 -- "mkdir -p gpurun_out; (for i in 1 2; do timeout -k 10 100 python3 _work/p/mcase.py \$PWD/_work/start $* && timeout -k 10 100 python3 _work/p/mcase.py \$PWD $* || exit 1; done) > gpurun_out/mc.log 2>&1; rc=\$?; exit \$rc" | grep "status="; grep pass gpurun_out/mc.log
